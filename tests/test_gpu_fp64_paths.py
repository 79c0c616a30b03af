"""The FP64 kernels at the sizes where their work splits change.

M2L per pair (k_m2l_fp64): orders whose outputs fill part of a wave, more
than one wave's lanes (P = 12, 16) and a single output range (P = 2), both
truncations, with few cells (lists shared out over workgroups) and many (one
workgroup per cell); P2P (k_p2p64): leaves of 1 .. ncrit bodies.  FP64 sums of
the same terms in another order: |diff| <= 1e-11 max |oracle|, the bar of the
parity tests.
"""
import numpy as np
import pytest

from minimal_amd import fmm
from minimal_amd.inputs import plummer, uniform_cube

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,P,full", [(200, 2, False), (200, 16, True), (2500, 3, True), (2500, 7, False),
                                      (2500, 12, False), (12000, 10, True), (12000, 9, False)])
def test_fp64_evaluation(gpu, orc, n, P, full):
    b0 = uniform_cube(n, n + P, "sym")
    b0["X"][: n // 2] = plummer(n // 2, 0.05, 0.5, np.random.default_rng(P))
    ref = b0.copy()
    orc.fmm(ref, P, 20, 0.5, full=full)
    f = fmm.FMM(P=P, ncrit=20, theta=0.5, m2l_precision=fmm.PREC_FP64, p2p_precision=fmm.PREC_FP64,
                m2l_truncation=fmm.M2L_FULL if full else fmm.M2L_REFERENCE)
    b = b0.copy()
    f.evaluate(b)
    assert np.array_equal(b["X"], ref["X"])
    for k in ("p", "F"):
        assert np.max(np.abs(b[k] - ref[k])) <= 1e-11 * np.max(np.abs(ref[k])), k
