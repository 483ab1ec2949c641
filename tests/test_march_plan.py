"""How the marching kernels split a volume's planes, on the CPU
(tests/cpp/march_plan_test.cpp, tipl_amd/csrc/march_plan.hpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_march_plan(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "march_plan_test")
    r = subprocess.run([gxx, "-std=c++17", "-O2", "-Wall", "-Wextra",
                        os.path.join(ROOT, "tests", "cpp", "march_plan_test.cpp"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "march plan ok" in r.stdout, r.stdout + r.stderr
