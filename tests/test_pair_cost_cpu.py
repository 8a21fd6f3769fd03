"""The choice between fused pairs and half-steps in place, against shapes that
were measured both ways (g++, no GPU; tests/cpp/pair_cost_selftest.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_pair_cost(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "pair_cost_selftest")
    subprocess.run([gxx, "-O2", "-std=c++17", "-Wall", "-pthread", f"-I{ROOT}/turbulent_lbm_multigpu_amd/csrc",
                    os.path.join(ROOT, "tests", "cpp", "pair_cost_selftest.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout
