"""Positions and capacities of the interaction lists around 2^31 entries, on
the CPU (tests/cpp/list_capacity.cxx)."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ missing")
def test_list_capacity(tmp_path):
    exe = str(tmp_path / "list_capacity")
    subprocess.run(["g++", "-std=c++17", "-O1", os.path.join(ROOT, "tests", "cpp", "list_capacity.cxx"), "-o", exe],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
