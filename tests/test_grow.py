"""Arrays that grow together keep their sizes in step through failed
allocations (tests/cpp/grow.cxx, on the CPU); on the device a context builds
trees of growing depth and size, among them a first build deeper than the prefix
histogram, whose cell arrays move after the root was written."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from conftest import ROOT
from minimal_amd import fmm
from minimal_amd.inputs import plummer, uniform_cube


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ missing")
def test_failed_allocations(tmp_path):
    exe = str(tmp_path / "grow")
    subprocess.run(["g++", "-std=c++17", "-O1", os.path.join(ROOT, "tests", "cpp", "grow.cxx"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


def _deep(n, a):
    b = uniform_cube(n, n, "sym")
    b["X"] = plummer(n, a, 0.5, np.random.default_rng(n))
    return b


@pytest.mark.gpu
@pytest.mark.parametrize("first", [0, 1])
def test_cells_after_growth(gpu, orc, first):
    sets = [uniform_cube(300, 1, "sym"), _deep(3000, 1e-4), uniform_cube(20000, 2, "sym"), _deep(30000, 1e-3),
            uniform_cube(50, 3, "sym")]
    f = fmm.FMM(P=4, ncrit=16, theta=0.4)
    for b0 in sets[first:]:
        s = orc.session(4, 16, 0.4)
        ref, b = b0.copy(), b0.copy()
        s.build_tree(ref)
        f.build_tree(b)
        assert np.array_equal(b["X"], ref["X"])
        c, r = f.cells(), s.cells()
        for k in ("nchild", "nbody", "child", "body", "X", "R"):
            assert np.array_equal(c[k], r[k]), k
