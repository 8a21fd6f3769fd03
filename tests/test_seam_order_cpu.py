"""Which wavefront takes which pair of a periodic row, on the CPU (g++, no GPU;
tests/cpp/seam_order_selftest.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_seam_order(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "seam_order_selftest")
    subprocess.run([gxx, "-O2", "-std=c++17", "-Wall", f"-I{ROOT}/turbulent_lbm_multigpu_amd/csrc",
                    os.path.join(ROOT, "tests", "cpp", "seam_order_selftest.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout
