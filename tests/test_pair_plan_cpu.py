"""The tiles of the fused beta + alpha kernel on the CPU (g++, no GPU): every
cell stored once, every gather inside the domain, every LDS neighbour computed
(tests/cpp/pair_plan_selftest.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_pair_plan(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "pair_plan_selftest")
    subprocess.run([gxx, "-O2", "-std=c++17", "-Wall", f"-I{ROOT}/turbulent_lbm_multigpu_amd/csrc",
                    os.path.join(ROOT, "tests", "cpp", "pair_plan_selftest.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout
