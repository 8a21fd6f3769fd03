"""The plan by which members that exchange faces run as fused pairs, on the
CPU (g++, no GPU): whole for the present members or empty
(tests/cpp/face_plan_selftest.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_face_plan(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "face_plan_selftest")
    subprocess.run([gxx, "-O2", "-std=c++17", "-Wall", "-D_GLIBCXX_ASSERTIONS",
                    f"-I{ROOT}/turbulent_lbm_multigpu_amd/csrc",
                    os.path.join(ROOT, "tests", "cpp", "face_plan_selftest.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout
