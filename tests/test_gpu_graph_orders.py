"""A grouped graph over problems of every order, small (the orders' P2M in one
launch) and larger (a launch per order): each replay against the same contexts
evaluated one by one.  Bar as for grouped graphs: relative L2 <= 1e-6 (the FP32
partial sums of M2L differ in order); bit-exact between replays."""
import numpy as np
import pytest

from minimal_amd import fmm
from minimal_amd.inputs import BODY_DTYPE, rel_l2, uniform_cube

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n", [300, 2500])
def test_every_order(gpu, n):
    devs, ctxs, eager = [], [], []
    for P in range(2, 17):
        b = uniform_cube(n + 7 * P, P, "unit_over_n")
        d = torch.from_numpy(b.view(np.uint8).copy()).cuda()
        torch.cuda.synchronize()
        f = fmm.FMM(P=P, ncrit=32, theta=0.5)
        f.evaluate(d.data_ptr(), n=len(b), on_device=True)
        f.synchronize()
        devs.append(d)
        ctxs.append(f)
        eager.append(d.cpu().numpy().view(BODY_DTYPE).copy())
    g = fmm.Graph(ctxs, grouped=True)
    first = None
    for _ in range(3):
        g.launch()
        g.synchronize()
        res = [d.cpu().numpy().view(BODY_DTYPE).copy() for d in devs]
        for P, r, e in zip(range(2, 17), res, eager):
            assert rel_l2(r["p"], e["p"]) <= 1e-6 and rel_l2(r["F"], e["F"]) <= 1e-6, P
        first = first or res
        assert all(np.array_equal(a["p"], b["p"]) and np.array_equal(a["F"], b["F"]) for a, b in zip(first, res))
        x = torch.ones(1 << 20, device="cuda").sum()
        assert float(x) == float(1 << 20)
    g.close()
