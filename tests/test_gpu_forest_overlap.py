"""Problems of a forest batch over one body array: the orders are evaluated one
after the other, lowest first, each adding to what the ones before left, as
separate calls would -- also once the shapes are tuned and forests without
shared bodies run side by side.  Bars as for a forest against its problems alone."""
import numpy as np
import pytest

from minimal_amd import fmm
from minimal_amd.inputs import BODY_DTYPE, rel_l2, uniform_cube

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

ORDERS = (12, 4, 8, 6)  # as given; evaluated 4, 6, 8, 12


def _reference(b0):
    b = b0.copy()
    for P in sorted(ORDERS):
        f = fmm.FMM(P=P, ncrit=32, theta=0.4)
        f.evaluate(b)
        f.close()
    return b


@pytest.mark.parametrize("device", [False, True])
def test_one_body_set_at_several_orders(gpu, device):
    f = fmm.FMM(ncrit=32, theta=0.4)
    for call in range(4):
        b0 = uniform_cube(30000, 5, "sym")
        if device:
            d = torch.from_numpy(b0.view(np.uint8).copy()).cuda()
            torch.cuda.synchronize()
            f.evaluate_batch([(d.data_ptr(), len(b0), P) for P in ORDERS], forest=True)
            b = d.cpu().numpy().view(BODY_DTYPE)
        else:
            b = b0.copy()
            f.evaluate_batch([(b, P) for P in ORDERS], forest=True)
        ref = _reference(b0)
        assert np.array_equal(b["X"], ref["X"]) and np.array_equal(b["q"], ref["q"])
        assert rel_l2(b["p"], ref["p"]) <= 2e-6 and rel_l2(b["F"], ref["F"]) <= 1e-5
