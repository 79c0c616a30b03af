"""The interaction lists where the traversal changes its way: targets whose
pairs overflow the small work queue (a pass repeated with the large one), lists
longer than the entries staged per target, key sets beyond the parallel
ranking (sorted by the radix sort), and contexts that repeat a pass and are
then used again.  The lists equal the oracle's as sets per target cell.
"""
import numpy as np
import pytest

from minimal_amd import fmm
from minimal_amd.inputs import plummer_background, rel_l2, uniform_cube

pytestmark = pytest.mark.gpu


def _same_lists(f, s):
    for which in (0, 1):
        off, src = f.lists(which)
        roff, rsrc = s.lists(which)
        assert np.array_equal(off, roff)
        for i in range(len(off) - 1):
            assert np.array_equal(np.sort(src[off[i]:off[i + 1]]), np.sort(rsrc[roff[i]:roff[i + 1]])), (which, i)


# largest queue / longest M2L list / longest hand-down list of a target:
# 200 / 195 / 80, then 835 / 549 / 420
@pytest.mark.parametrize("n,ncrit,theta", [(1500, 4, 0.4), (3000, 6, 0.2)])
def test_lists(gpu, orc, n, ncrit, theta):
    s = orc.session(4, ncrit, theta)
    b = uniform_cube(n, 1, "sym")
    s.build_tree(b)
    s.make_lists()
    f = fmm.FMM(P=4, ncrit=ncrit, theta=theta)
    for _ in range(2):
        b = uniform_cube(n, 1, "sym")
        f.build_tree(b)
        f.upward()
        f.horizontal()
        _same_lists(f, s)


def test_key_set_beyond_ranking(gpu):
    """14,132 keys: the keyed GEMM on the radix-sorted numbering against the
    FP64 M2L per pair (charges of one sign; the BF16x3 bar of a same-signed
    sum, 3 x 2^-17)."""
    b0 = plummer_background(50000, 1)
    b0["q"] = np.abs(b0["q"]) / len(b0)
    out = []
    for prec in (fmm.PREC_BF16X3, fmm.PREC_FP64):
        f = fmm.FMM(P=4, ncrit=8, theta=0.25, m2l_precision=prec)
        b = b0.copy()
        f.evaluate(b)
        assert f.work_counts()["m2l_keys"] > 12288
        out.append(b)
        f.close()
    assert rel_l2(out[0]["p"], out[1]["p"]) <= 3 * 2.0 ** -17
