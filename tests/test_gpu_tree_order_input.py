"""Trees of bodies that come in tree order, as a time-stepping program's do:
neighbouring bodies share their prefixes, in runs that cross wave boundaries, end
in partly filled waves, and mix with single ones.  Bit-exact against the oracle on
the same input, for the first build of a context and the builds after it."""
import numpy as np
import pytest

from minimal_amd import fmm
from minimal_amd.inputs import plummer, uniform_cube

pytestmark = pytest.mark.gpu


def _input(kind, n, orc, ncrit):
    b = uniform_cube(n, n, "sym")
    if kind == "clustered":
        b["X"] = plummer(n, 0.1, 0.5, np.random.default_rng(n))
    s = orc.session(2, ncrit, 0.4)
    s.build_tree(b)  # now in tree order
    if kind == "mixed":  # half of the bodies back among the others
        rng = np.random.default_rng(1)
        i = rng.permutation(n)[: n // 2]
        b[np.sort(i)] = b[i]
    return b


@pytest.mark.parametrize("kind", ["uniform", "clustered", "mixed"])
@pytest.mark.parametrize("n,ncrit", [(63, 8), (64, 8), (65, 64), (5001, 16), (40037, 300), (100000, 1024)])
def test_tree_order(gpu, orc, kind, n, ncrit):
    f = fmm.FMM(P=2, ncrit=ncrit, theta=0.4)
    b0 = _input(kind, n, orc, ncrit)
    for _ in range(2):
        b, ref = b0.copy(), b0.copy()
        s = orc.session(2, ncrit, 0.4)
        s.build_tree(ref)
        f.build_tree(b)
        assert np.array_equal(b["X"], ref["X"]) and np.array_equal(b["q"], ref["q"])
        c, r = f.cells(), s.cells()
        for k in ("nchild", "nbody", "child", "body", "X", "R"):
            assert np.array_equal(c[k], r[k]), k


@pytest.mark.parametrize("n,ncrit", [(760001, 300), (1600000, 64)])
def test_large_sets_by_either_sort(gpu, orc, n, ncrit):
    """Sizes that are sorted by radix or by counting, by the order in which the
    last build's bodies came: random, tree order twice (the second by counting),
    random on a hint of tree order, random again.  A tree built on its own order
    leaves the bodies where they are."""
    b0 = uniform_cube(n, 9, "sym")
    s = orc.session(2, ncrit, 0.4)
    ref = b0.copy()
    s.build_tree(ref)
    r = s.cells()
    f = fmm.FMM(P=2, ncrit=ncrit, theta=0.4)
    b = None
    for fresh in (True, False, False, True, True):
        b = b0.copy() if fresh else b
        f.build_tree(b)
        assert np.array_equal(b["X"], ref["X"]) and np.array_equal(b["q"], ref["q"])
        c = f.cells()
        for k in ("nchild", "nbody", "child", "body", "X", "R"):
            assert np.array_equal(c[k], r[k]), k
