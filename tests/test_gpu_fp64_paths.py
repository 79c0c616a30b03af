"""The FP64 kernels at the sizes where their work splits change.

M2L per pair (k_m2l_fp64): orders whose outputs fill part of a wave, more
than one wave's lanes (P = 12, 16) and a single output range (P = 2), both
truncations, with few cells (lists shared out over workgroups) and many (one
workgroup per cell); P2P (k_p2p64): leaves of 1 .. ncrit bodies.  FP64 sums of
the same terms in another order: |diff| <= 1e-11 max |oracle|, the bar of the
parity tests.

Direct sum (k_direct): one target, target blocks that are not full, one to
four blocks per workgroup, one launch and two, fewer sources than a wave, sources that coincide
with targets, and squared distances beyond the range of the fast 1/sqrt
(zero, denormal, overflowing).  Each interaction carries a few roundings of
2^-53 and n of them are added: |diff| <= (n + 16) 2^-53 sum |q / r|.
"""
import numpy as np
import pytest

from minimal_amd import fmm
from minimal_amd.inputs import BODY_DTYPE, plummer, uniform_cube

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


def _direct_reference(t, s):
    d = t["X"][:, None, :] - s["X"][None, :, :]
    with np.errstate(all="ignore"):
        r = np.sqrt((d.astype(np.longdouble) ** 2).sum(2))
        w = np.where(r > 0, s["q"] / np.where(r > 0, r, 1), 0)
        g = -(w / np.where(r > 0, r * r, 1))[:, :, None] * d
    return w.sum(1), g.sum(1), np.abs(w).sum(1), np.abs(g).sum(1)


@pytest.mark.parametrize("nt,ns", [(1, 1), (1, 3000), (7, 63), (9, 129), (33, 1000), (257, 4097)])
def test_direct_sum(gpu, nt, ns):
    s = uniform_cube(ns, 3 * ns + nt, "sym")
    t = uniform_cube(nt, 11, "sym")
    t["X"][::2] = s["X"][np.arange(len(t["X"][::2])) % ns]  # zero distances
    f = fmm.FMM()
    f.direct(t, s)
    p, F, ap, aF = _direct_reference(t, s)
    assert np.all(np.abs(t["p"] - p) <= (ns + 16) * 2.0 ** -53 * ap)
    assert np.all(np.abs(t["F"] - F) <= (ns + 16) * 2.0 ** -53 * aF)


def test_direct_sum_extreme_distances(gpu):
    """Squared distances 0, denormal, near the ends of the exponent range and
    overflowing (1/r is then 0, as 1 / inf).  A denormal r^2 holds few bits:
    compared with the same arithmetic in double."""
    x = np.array([0.0, 1e-160, 3e-155, 1e-130, 1e-100, 1.0, 1e100, 1e130, 1e154, 1e200])
    s = np.zeros(len(x), BODY_DTYPE)
    s["X"][:, 0] = x
    s["q"] = np.linspace(1, 2, len(x))
    f = fmm.FMM()
    for i in range(len(x)):
        t = np.zeros(1, BODY_DTYPE)
        f.direct(t, s[i:i + 1])
        r2 = x[i] * x[i]
        with np.errstate(all="ignore"):
            p = s["q"][i] * np.sqrt(1.0 / r2) if r2 != 0 else 0.0
        if np.isfinite(p):
            assert abs(t["p"][0] - p) <= 8 * 2.0 ** -53 * abs(p), (x[i], t["p"][0], p)
        else:
            assert not np.isfinite(t["p"][0])


@pytest.mark.parametrize("ns", [8192, 8193])
def test_direct_sum_launch_split(gpu, ns):
    """The most sources that one launch adds, and the fewest of two."""
    test_direct_sum(gpu, 3, ns)
