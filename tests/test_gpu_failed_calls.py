"""A call that fails leaves no half-made state: the passes after it report that
there is no tree (or no lists) instead of running on arrays and sizes of two
different body sets, and the context evaluates the next set as a new one does."""
import numpy as np
import pytest

from minimal_amd import fmm
from minimal_amd.inputs import uniform_cube

pytestmark = pytest.mark.gpu


def _fresh(n):
    b = uniform_cube(n, n, "sym")
    f = fmm.FMM(P=6, ncrit=16)
    f.evaluate(b)
    f.close()
    return b


@pytest.mark.parametrize("call", ["build_tree", "evaluate"])
def test_failed_build(gpu, call):
    f = fmm.FMM(P=6, ncrit=16)
    b = uniform_cube(2000, 2000, "sym")
    f.evaluate(b)
    bad = uniform_cube(9000, 1, "sym")
    bad["X"][17, 2] = np.nan
    with pytest.raises(fmm.ExaFMMError, match="non-finite"):
        getattr(f, call)(bad)
    for later in (f.upward, f.horizontal, f.downward, f.num_cells, f.work_counts, lambda: f.lists(0)):
        with pytest.raises(fmm.ExaFMMError) as e:
            later()
        assert e.value.code == -2  # EXAFMM_ERR_STATE
    b = uniform_cube(3000, 3000, "sym")
    f.evaluate(b)
    ref = _fresh(3000)
    assert np.array_equal(b["X"], ref["X"])
    # the same kernels; the tuned GEMM shape and so its sums' order may differ
    assert np.max(np.abs(b["p"] - ref["p"])) <= 1e-5 * np.max(np.abs(ref["p"]))


def test_failed_horizontal(gpu):
    """A horizontal pass that fails (pairs beyond the traversal's work queue)
    leaves the last one's locals and lists to no later call."""
    def tree(n):
        f = fmm.FMM(P=4, ncrit=4, theta=0.05, m2l_precision=fmm.PREC_FP64)
        f.build_tree(uniform_cube(n, 5, "sym"))
        f.upward()
        return f
    ft, fs = tree(60), tree(20000)
    ft.horizontal()
    with pytest.raises(fmm.ExaFMMError):
        ft.horizontal(fs)
    for later in (ft.downward, ft.work_counts):
        with pytest.raises(fmm.ExaFMMError) as e:
            later()
        assert e.value.code == -2
    ft.horizontal()
    ft.downward()
