"""The keyed BF16x3 GEMM at the sizes where its work split changes, against
the FP64 M2L per pair on the same tree: orders with one row tile (P = 2), k-steps
that a round cuts (P = 12), a full set of accumulators (P = 11, 12), two row
blocks of unequal height (P = 13, 15, 16); per-tile and stream-K launches; tiles
that are nearly empty (small trees of many levels), span several mask blocks of
64 keys, and hold several levels.

Tolerance: a product of hi + lo splits drops lo x lo and rounds lo (2^-17
relative each, three products), so a sum of same-signed terms is off by at
most 3 x 2^-17; charges of one sign keep the potential such a sum.  The force
sums terms of both signs, whose magnitudes exceed the result several times:
8 x 3 x 2^-17.
"""
import numpy as np
import pytest

from minimal_amd import fmm
from minimal_amd.inputs import plummer_background, rel_l2, uniform_cube

pytestmark = pytest.mark.gpu

BOUND = 3 * 2.0 ** -17


def _pair(b0, P, ncrit, **kw):
    out = []
    for prec in (fmm.PREC_BF16X3, fmm.PREC_FP64):
        f = fmm.FMM(P=P, ncrit=ncrit, theta=0.4, m2l_precision=prec, p2p_precision=fmm.PREC_FP64, **kw)
        b = b0.copy()
        f.evaluate(b)
        out.append(b)
        f.close()
    return out


@pytest.mark.parametrize("schedule", ["EXAFMM_GEMM_SK_ONLY", "EXAFMM_GEMM_NO_SK"])
@pytest.mark.parametrize("P", [2, 4, 6, 7, 8, 9, 11, 12, 13, 15, 16])
def test_orders(gpu, monkeypatch, P, schedule):
    monkeypatch.setenv(schedule, "1")
    b0 = plummer_background(6000, P)
    b0["q"] = np.abs(b0["q"]) / len(b0)
    fast, ref = _pair(b0, P, 16)
    assert np.array_equal(fast["X"], ref["X"])
    assert rel_l2(fast["p"], ref["p"]) <= BOUND
    assert rel_l2(fast["F"], ref["F"]) <= 8 * BOUND


@pytest.mark.parametrize("n,ncrit,images", [(600, 4, 0), (40000, 8, 0), (3000, 8, 2)])
def test_tile_fill(gpu, n, ncrit, images):
    b0 = uniform_cube(n, n, "unit_over_n")
    fast, ref = _pair(b0, 10, ncrit, images=images, cycle=1.0 if images else 0.0)
    assert rel_l2(fast["p"], ref["p"]) <= BOUND
    assert rel_l2(fast["F"], ref["F"]) <= 8 * BOUND
