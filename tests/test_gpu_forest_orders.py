"""Batches of more orders than forests run side by side: the first call runs
them in turn (GEMM shapes are tuned alone on the device), later calls on host
threads, also with other problem sizes, whose shapes are tuned by the call
after; a forest that fails reports its error and the others' problems and the
context stay usable.  Bars as for a forest against its problems alone.
"""
import numpy as np
import pytest

from minimal_amd import fmm
from minimal_amd.inputs import plummer, rel_l2, uniform_cube

pytestmark = pytest.mark.gpu

ORDERS = (3, 4, 6, 7, 8, 10)


def _problems(scale, seed):
    out = []
    for i in range(2 * len(ORDERS)):
        n = scale * (200 + 37 * i)
        b = uniform_cube(n, seed + i, "sym")
        if i % 2:
            b["X"] = plummer(n, 0.05, 0.5, np.random.default_rng(seed + i))
        out.append((b, ORDERS[i % len(ORDERS)]))
    return out


def _check(f, scale, seed):
    probs = _problems(scale, seed)
    ref = [(b.copy(), P) for b, P in probs]
    f.evaluate_batch(probs, forest=True)
    for (b, P), (r, _) in zip(probs, ref):
        g = fmm.FMM(P=P, ncrit=32, theta=0.4)
        g.evaluate(r)
        g.close()
        assert np.array_equal(b["X"], r["X"]) and np.array_equal(b["q"], r["q"])
        assert rel_l2(b["p"], r["p"]) <= 2e-6 and rel_l2(b["F"], r["F"]) <= 1e-5


def test_repeated_batches(gpu):
    f = fmm.FMM(ncrit=32, theta=0.4)
    for scale, seed in ((1, 1), (1, 50), (12, 100), (12, 150), (3, 200)):
        _check(f, scale, seed)


def test_failing_forest(gpu):
    f = fmm.FMM(ncrit=32, theta=0.4)
    _check(f, 1, 1)
    probs = _problems(1, 300)
    probs[2][0]["X"][5, 1] = np.nan
    with pytest.raises(fmm.ExaFMMError, match="non-finite"):
        f.evaluate_batch(probs, forest=True)
    _check(f, 1, 2)
