"""The FP32 keyed GEMM over the orders (one row block and several, remainders of
the row tiles and k-steps), on tiles with empty subtiles, with key slices, in
periodic trees and with learned orders, against the FP64 M2L per pair on the same
tree.

Tolerance: products and sums of 24-bit numbers; a column's accumulator adds a few
hundred keys' terms, whose roundings add like a random walk of that length: below
64 x 2^-24 for the potential of charges of one sign, eight times that for the
force (terms of both signs).
"""
import numpy as np
import pytest

from minimal_amd import fmm
from minimal_amd.inputs import plummer_background, rel_l2, uniform_cube

pytestmark = pytest.mark.gpu

BOUND = 64 * 2.0 ** -24


def _check(b0, **kw):
    out = []
    for prec in (fmm.PREC_FP32, fmm.PREC_FP64):
        f = fmm.FMM(m2l_precision=prec, p2p_precision=fmm.PREC_FP64, **kw)
        for _ in range(2):  # the second run takes the tuned shape
            b = b0.copy()
            f.evaluate(b)
        out.append(b)
        f.close()
    assert np.array_equal(out[0]["X"], out[1]["X"])
    assert rel_l2(out[0]["p"], out[1]["p"]) <= BOUND
    assert rel_l2(out[0]["F"], out[1]["F"]) <= 8 * BOUND


@pytest.mark.parametrize("P", range(2, 17))
def test_orders(gpu, P):
    b0 = plummer_background(6000, P)
    b0["q"] = np.abs(b0["q"]) / len(b0)
    _check(b0, P=P, ncrit=16, theta=0.4)


@pytest.mark.parametrize("n,ncrit,theta", [(100, 4, 0.5), (3000, 8, 0.3), (60000, 32, 0.4)])
def test_tile_fill(gpu, n, ncrit, theta):
    _check(uniform_cube(n, n, "unit_over_n"), P=9, ncrit=ncrit, theta=theta)


def test_periodic(gpu):
    _check(uniform_cube(5000, 3, "unit_over_n"), P=8, ncrit=16, theta=0.4, images=2, cycle=1.0)


def test_learned_orders(gpu):
    """Orders of their own per key: against BF16x3 on the same tree and model, within
    that form's bar (3 x 2^-17)."""
    b0 = plummer_background(20000, 8)
    b0["q"] = np.abs(b0["q"]) / len(b0)
    t = fmm.FMM(P=14, ncrit=64, theta=0.4)  # (the order that training needs)
    t.build_tree(b0.copy())
    t.upward()
    t.horizontal()
    t.train_order_model(nsamples=2048, epochs=20)
    w = t.order_model()
    t.close()
    out = []
    for prec in (fmm.PREC_FP32, fmm.PREC_BF16X3):
        f = fmm.FMM(P=12, ncrit=64, theta=0.4, m2l_precision=prec, order_policy=fmm.ORDER_LEARNED)
        f.set_order_model(w, -5.0)
        b = b0.copy()
        f.evaluate(b)
        assert np.count_nonzero(f.order_stats()) > 1
        out.append(b)
        f.close()
    assert rel_l2(out[0]["p"], out[1]["p"]) <= 3 * 2.0 ** -17
    assert rel_l2(out[0]["F"], out[1]["F"]) <= 8 * 3 * 2.0 ** -17
