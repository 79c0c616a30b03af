"""Forests run side by side on no more host threads than the calling thread has
CPUs, and none where EXAFMM_FOREST_THREADS asks for one at a time; the results
are the same."""
import os
import threading

import numpy as np
import pytest

from minimal_amd import fmm
from minimal_amd.inputs import rel_l2, uniform_cube

pytestmark = pytest.mark.gpu

ORDERS = (4, 6, 8, 10)


class _Sampler(threading.Thread):
    """Largest number of threads of this process while it runs."""

    def __init__(self):
        super().__init__(daemon=True)
        self.stop, self.most = False, 0

    def run(self):
        os.sched_setaffinity(0, self.cpus)
        while not self.stop:
            self.most = max(self.most, len(os.listdir("/proc/self/task")))


def _threads(f, calls=30):
    s = _Sampler()
    s.cpus = ALL
    s.start()
    before = len(os.listdir("/proc/self/task"))
    for _ in range(calls):
        probs = [(uniform_cube(3000, P, "sym"), P) for P in ORDERS]
        f.evaluate_batch(probs, forest=True)
    s.stop = True
    s.join()
    return s.most - before, probs


ALL = os.sched_getaffinity(0)


@pytest.mark.parametrize("how", ["one cpu", "environment"])
def test_no_threads(gpu, monkeypatch, how):
    f = fmm.FMM(ncrit=32, theta=0.4)
    for _ in range(4):  # tuned
        f.evaluate_batch([(uniform_cube(3000, P, "sym"), P) for P in ORDERS], forest=True)
    ref = _threads(f)[1]
    try:
        if how == "one cpu":
            os.sched_setaffinity(0, {min(ALL)})
        else:
            monkeypatch.setenv("EXAFMM_FOREST_THREADS", "1")
        more, probs = _threads(f)
    finally:
        os.sched_setaffinity(0, ALL)
    assert more == 0
    for (a, _), (b, _) in zip(probs, ref):
        assert np.array_equal(a["X"], b["X"]) and rel_l2(a["p"], b["p"]) <= 2e-6
