"""P2M and L2P at every order: their loops over the degrees are unrolled per
order, lanes hold columns in pairs (odd orders leave one alone), and leaves of
one body, of a few, of a wave's share and of several lie in one tree.

Multipoles are FP64 sums of the same terms in another order: 1e-12 (the bar of
the parity tests) of the terms' sum, |Y_n^m| <= rho^n / n!, with the distances
of a leaf's bodies and the half diagonal of a larger cell.
"""
import math

import numpy as np
import pytest

from minimal_amd import fmm
from minimal_amd.inputs import plummer, rel_l2, uniform_cube

pytestmark = pytest.mark.gpu


def _bodies(n, seed):
    b = uniform_cube(n, seed, "sym")
    b["X"][: n // 2] = plummer(n // 2, 0.05, 0.5, np.random.default_rng(seed))
    return b


@pytest.mark.parametrize("P", range(2, 17))
@pytest.mark.parametrize("n,ncrit", [(1, 64), (3000, 100)])
def test_multipoles(gpu, orc, P, n, ncrit):
    b, b2 = _bodies(n, 7 * P + n), _bodies(n, 7 * P + n)
    s = orc.session(P, ncrit, 0.4)
    s.build_tree(b2)
    s.upward(b2)
    f = fmm.FMM(P=P, ncrit=ncrit, theta=0.4)
    f.build_tree(b)
    f.upward()
    cells, diff = f.cells(), np.abs(f.multipoles() - s.M())
    for i, c in enumerate(cells):
        mine = b[c["body"]:c["body"] + c["nbody"]]
        rho = np.linalg.norm(mine["X"] - c["X"], axis=1) if c["nchild"] == 0 else 3 ** 0.5 * c["R"]
        for k in range(P):
            bound = np.sum(np.abs(mine["q"]) * rho ** k) / math.factorial(k)
            assert np.all(diff[i, k * (k + 1) // 2:(k + 1) * (k + 2) // 2] <= 1e-12 * bound), (i, k)


@pytest.mark.parametrize("P", range(2, 17))
@pytest.mark.parametrize("n,ncrit", [(2000, 2), (3000, 100)])
def test_field(gpu, orc, P, n, ncrit):
    """Leaves of one or two bodies (many runs of equal leaf per wave) and of
    up to a hundred: parity mode against the oracle at its bar, FP32 M2L and
    L2P within the bar of the FP32 path."""
    b0 = _bodies(n, 5 * P)
    ref = b0.copy()
    orc.fmm(ref, P, ncrit, 0.4, full=True)
    for prec, bar in ((fmm.PREC_FP64, 1e-11), (fmm.PREC_FP32, 3e-6)):
        f = fmm.FMM(P=P, ncrit=ncrit, theta=0.4, m2l_precision=prec, p2p_precision=fmm.PREC_FP64,
                    m2l_truncation=fmm.M2L_FULL)
        b = b0.copy()
        f.evaluate(b)
        for k in ("p", "F"):
            assert rel_l2(b[k], ref[k]) <= bar, (prec, k)


@pytest.mark.parametrize("P", [12, 14])
def test_wide_levels(gpu, P):
    """Levels of more cells than a workgroup of the L2L pass lists at a time
    (1,024 in each of 32 ranges; order 14 takes two passes over its row
    tiles), against the direct sum at the truncation error of the order."""
    b0 = uniform_cube(60000, P, "sym")
    f = fmm.FMM(P=P, ncrit=1, theta=0.35)
    f.evaluate(b0)
    assert f.num_cells()[0] > 2 * 32768
    t = b0[:: len(b0) // 2000].copy()
    fp, fF = t["p"].copy(), t["F"].copy()
    t["p"], t["F"] = 0, 0
    f.direct(t, b0)
    assert rel_l2(fp, t["p"]) <= 1e-5
    assert rel_l2(fF, t["F"]) <= 1e-5
