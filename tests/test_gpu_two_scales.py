"""FP64 M2L between trees of very different size: a target tree 10^9 to 10^80
times smaller (near the origin) than the sources.  The powers of the ratio of the
radii leave the range of double long before their products do.

Bar against the direct sum: the targets are a point at the sources' scale, so
that only the sources' expansions are cut, whose terms fall like 0.3^n at theta =
0.3, with both signs among the bodies of a cell: 1e-6 of max |p| at P = 10 and 16,
ten times that for the force; at P = 2 that the value is of the right size.
"""
import numpy as np
import pytest

from minimal_amd import fmm
from minimal_amd.inputs import uniform_cube

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,full", [(10, True), (16, True), (16, False), (2, True)])
@pytest.mark.parametrize("scale", [1e-9, 1e-18, 1e-22, 1e-40, 1e-80])
def test_scales(gpu, P, full, scale):
    t = uniform_cube(100, 1, "sym")
    t["X"] *= scale
    t["p"] = 0
    s = uniform_cube(3000, 2, "unit_over_n")
    s["X"] += 1.5
    mk = lambda: fmm.FMM(P=P, ncrit=16, theta=0.3, m2l_truncation=fmm.M2L_FULL if full else fmm.M2L_REFERENCE,
                         m2l_precision=fmm.PREC_FP64, p2p_precision=fmm.PREC_FP64)
    ft, fs = mk(), mk()
    ft.build_tree(t)
    fs.build_tree(s)
    fs.upward()
    ft.horizontal(fs)
    assert ft.work_counts()["m2l_pairs"] > 0
    ft.downward()
    d = t["X"][:, None] - s["X"][None]
    r2 = (d * d).sum(2)
    w = s["q"] / np.sqrt(r2)
    p, F = w.sum(1), -((w / r2)[:, :, None] * d).sum(1)
    bar = 1e-6 if P > 2 else 0.3
    assert np.max(np.abs(t["p"] - p)) <= bar * np.max(np.abs(p))
    assert np.max(np.abs(t["F"] - F)) <= 10 * bar * np.max(np.abs(F))
