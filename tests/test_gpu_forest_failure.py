"""A batch of forests that fails returns with every forest's work ended: the
problems of the forests that did not fail hold their results and no kernel or
copy writes to them any more."""
import time

import numpy as np
import pytest

from minimal_amd import fmm
from minimal_amd.inputs import BODY_DTYPE, uniform_cube

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("tuned", [False, True])
def test_no_work_after_the_error(gpu, tuned):
    f = fmm.FMM(ncrit=64, theta=0.4)
    sets = [(uniform_cube(400000, 1, "sym"), 6), (uniform_cube(400000, 2, "sym"), 8), (uniform_cube(500, 3, "sym"), 10)]

    def call(fail):
        devs = []
        for b, P in sets:
            h = b.copy()
            if fail and P == 10:
                h["X"][7, 0] = np.nan
            devs.append(torch.from_numpy(h.view(np.uint8).copy()).cuda())
        torch.cuda.synchronize()
        probs = [(d.data_ptr(), len(b), P) for d, (b, P) in zip(devs, sets)]
        if not fail:
            f.evaluate_batch(probs, forest=True)
            return devs, None
        now = [d.clone() for d in devs[:2]]
        s = torch.cuda.Stream()  # waits for none of the library's
        torch.cuda.synchronize()
        try:
            f.evaluate_batch(probs, forest=True)
            failed = False
        except fmm.ExaFMMError as e:
            with torch.cuda.stream(s):
                for n, d in zip(now, devs):
                    n.copy_(d)
            s.synchronize()
            failed = "non-finite" in str(e)
        assert failed
        return devs, now

    if tuned:  # the forests then run side by side
        for _ in range(3):
            good, _ = call(False)
    devs, now = call(True)
    time.sleep(0.2)
    torch.cuda.synchronize()
    for d, n in zip(devs, now):
        assert torch.equal(d, n)
        assert np.any(d.cpu().numpy().view(BODY_DTYPE)["p"] != 0)
