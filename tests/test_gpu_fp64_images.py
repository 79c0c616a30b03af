"""FP64 P2P across periodic images: dX = Xi - Xj - iX * cycle with the image
shift subtracted last (3dp/kernel.h:133), so that pairs at zero distance through
an image are those of that arithmetic.  0.3 - (-0.7) rounds to the cycle of 1:
the pair is skipped, where -0.7 + 1 is 0.3 plus half a unit in the last place and
would count as a pair at a distance of 6e-17.

Bar: the same sum in double by numpy, 54 terms of a few roundings each:
64 x 2^-53 of the sum of magnitudes.
"""
import numpy as np
import pytest

from minimal_amd import fmm
from minimal_amd.inputs import BODY_DTYPE, uniform_cube

pytestmark = pytest.mark.gpu


def _sum(b, cycle):
    p, F, ap, aF = np.zeros(len(b)), np.zeros((len(b), 3)), np.zeros(len(b)), np.zeros((len(b), 3))
    for img in range(27):
        sh = np.array([img % 3 - 1, img // 3 % 3 - 1, img // 9 - 1]) * cycle
        d = b["X"][:, None] - b["X"][None] - sh
        r2 = (d * d).sum(2)
        w = np.where(r2 != 0, b["q"] / np.sqrt(np.where(r2 != 0, r2, 1)), 0)
        g = (w / np.where(r2 != 0, r2, 1))[:, :, None] * d
        p += w.sum(1)
        F -= g.sum(1)
        ap += np.abs(w).sum(1)
        aF += np.abs(g).sum(1)
    return p, F, ap, aF


@pytest.mark.parametrize("case", ["meet", "random"])
def test_images(gpu, case):
    if case == "meet":
        b = np.zeros(4, BODY_DTYPE)
        b["X"] = [[0.3, 0.1, 0.2], [-0.7, 0.1, 0.2], [0.1, 0.3, -0.7], [0.1, -0.7, 0.3]]
        b["q"] = [1.0, 2.0, 0.5, 0.25]
        assert b["X"][0, 0] - b["X"][1, 0] - 1.0 == 0.0 and b["X"][0, 0] - (b["X"][1, 0] + 1.0) != 0.0
    else:
        b = uniform_cube(60, 5, "sym")
        b["X"] = np.round(b["X"] * 16) / 16 - 0.5
    f = fmm.FMM(P=4, ncrit=64, theta=0.4, images=1, cycle=1.0, m2l_precision=fmm.PREC_FP64,
                p2p_precision=fmm.PREC_FP64)
    f.evaluate(b)
    assert f.work_counts()["m2l_pairs"] == 0  # the root alone: every image by P2P
    p, F, ap, aF = _sum(b, 1.0)
    tol = (27 * len(b) + 10) * 2.0 ** -53
    assert np.all(np.abs(b["p"] - p) <= tol * ap)
    assert np.all(np.abs(b["F"] - F) <= tol * aF)
