"""A traversal whose lists outgrow their room is repeated with more: a few
target cells in small groups against a fine source tree at theta = 0.2 hand down
more pairs than the first pass has room for (96 per cell), at a level with more
levels below it, and overflow the small work queue as well.  The lists and FP64
results equal those of a context whose lists have room from the start (it held a
larger tree before), bit for bit.
"""
import numpy as np
import pytest

from minimal_amd import fmm
from minimal_amd.inputs import BODY_DTYPE, uniform_cube

pytestmark = pytest.mark.gpu


def _targets(groups=16, n=6, size=0.005):
    rng = np.random.default_rng(1)
    b = np.zeros(8 + groups * n, BODY_DTYPE)
    b["X"][:8] = [[i & 1, i >> 1 & 1, i >> 2 & 1] for i in range(8)]
    c = 0.3 + 0.4 * rng.random((groups, 3))
    b["X"][8:] = np.repeat(c, n, 0) + rng.random((groups * n, 3)) * size
    b["q"] = rng.random(len(b))
    return b


def _sources(n=2000):
    b = uniform_cube(n, 2, "sym")
    b["X"] = 0.2 + 0.6 * b["X"]
    return b


def _context(b, ncrit):
    f = fmm.FMM(P=6, ncrit=ncrit, theta=0.2, m2l_precision=fmm.PREC_FP64, p2p_precision=fmm.PREC_FP64)
    f.build_tree(b)
    f.upward()
    return f


def test_hand_down_list_grows(gpu):
    src = _sources()
    fs = _context(src, 2)
    out = []
    for before in (False, True):
        t = _targets()
        if before:
            f = _context(uniform_cube(8000, 3, "sym"), 4)
            f.horizontal()
            f.build_tree(t)
            f.upward()
        else:
            f = _context(t, 4)
        f.horizontal(fs)
        assert f.work_counts()["cells"] * 96 < 17999  # pairs handed down in all
        f.downward()
        out.append((t, f.lists(0), f.lists(1)))
        f.close()
    (a, am, ap), (b, bm, bp) = out
    for x, y in ((am, bm), (ap, bp)):
        assert np.array_equal(x[0], y[0]) and np.array_equal(x[1], y[1])
    assert np.array_equal(a["p"], b["p"]) and np.array_equal(a["F"], b["F"])
    # all of the pairs are there (the expansions' error is far below)
    ref = np.array([(src["q"] / np.linalg.norm(src["X"] - x, axis=1)).sum() for x in a["X"]])
    assert np.max(np.abs(a["p"] - ref)) <= 1e-3 * np.max(np.abs(ref))
