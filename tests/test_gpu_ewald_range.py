"""The Ewald sum's pair function at the ends of the exponent range: distances
whose squares are denormal (the potential is finite, 1/r), and alpha r whose
square is near the largest double or beyond (the potential is 0; the force's
factor alpha^3 leaves the range of double before that, above 1e102).  Bar: a denormal
square holds few bits: against the same double arithmetic, q / sqrt(r^2), 8 x
2^-53."""
import numpy as np
import pytest

from minimal_amd import fmm
from minimal_amd.inputs import BODY_DTYPE

pytestmark = pytest.mark.gpu


def _pair(x, alpha):
    s, t = np.zeros(1, BODY_DTYPE), np.zeros(1, BODY_DTYPE)
    s["q"] = 1.0
    t["X"][0] = x, 0.0, 0.0
    f = fmm.FMM(images=2, cycle=400.0)
    f.ewald(t, s, 0, alpha, 0.25 / np.pi, 100.0)
    return t[0]


@pytest.mark.parametrize("x", [1e-120, 1e-140, 1e-154, 1e-157, 1e-160])
def test_small(gpu, x):
    p = 1.0 / np.sqrt(x * x)
    assert abs(_pair(x, 1.0)["p"] - p) <= 8 * 2.0 ** -53 * p


@pytest.mark.parametrize("alpha", [1e100, 1e140, 9e153, 1e154, 1e160])
def test_large(gpu, alpha):
    t = _pair(1.0, alpha)
    assert t["p"] == 0.0
    if alpha <= 1e100:
        assert np.all(t["F"] == 0.0)
