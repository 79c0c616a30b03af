"""The direct and Ewald sums on either side of the sizes where the workgroups'
shape changes: few sources, many targets, both.  Against long double, with the
bars of the sums' other tests: (ns + 16) 2^-53 of the sum of magnitudes, and 1e-11
of the largest value."""
import numpy as np
import pytest

from minimal_amd import fmm
from minimal_amd.inputs import uniform_cube
from test_gpu_ewald_edges import SIGMA, _reference
from test_gpu_fp64_paths import _direct_reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt,ns", [(30, 512), (30, 513), (1999, 600), (2000, 600), (2003, 2500), (5001, 17)])
def test_direct(gpu, nt, ns):
    s, t = uniform_cube(ns, ns, "sym"), uniform_cube(nt, nt, "sym")
    fmm.FMM().direct(t, s)
    for a in range(0, nt, 500):
        p, F, ap, aF = _direct_reference(t[a:a + 500], s)
        assert np.all(np.abs(t["p"][a:a + 500] - p) <= (ns + 16) * 2.0 ** -53 * ap)
        assert np.all(np.abs(t["F"][a:a + 500] - F) <= (ns + 16) * 2.0 ** -53 * aF)


@pytest.mark.parametrize("nt,ns,ksize", [(1024, 50, 3), (1025, 50, 3), (1025, 256, 2), (1027, 257, 2), (1030, 40, 7),
                                         (1500, 700, 4)])
def test_ewald(gpu, nt, ns, ksize):
    cyc, alpha, cutoff = 1.3, 7.0, 0.5
    s, t = uniform_cube(ns, 3 * ns, "sym"), uniform_cube(nt, nt, "sym")
    s["X"] *= cyc
    t["X"] *= cyc
    f = fmm.FMM(images=2, cycle=cyc)
    f.ewald(t, s, ksize, alpha, SIGMA, cutoff)
    for a in range(0, nt, 500):
        p, F = _reference(t[a:a + 500], s, ksize, alpha, cutoff, cyc)
        assert np.max(np.abs(t["p"][a:a + 500] - p)) <= 1e-11 * np.max(np.abs(p))
        assert np.max(np.abs(t["F"][a:a + 500] - F)) <= 1e-11 * np.max(np.abs(F))
