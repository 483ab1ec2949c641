"""Which volumes take the CDM kernels with 32-bit byte offsets, on the CPU
(tests/cpp/field_limits_test.cpp, tipl_amd/csrc/field_limits.hpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_field_limits(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "field_limits_test")
    r = subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Wextra",
                        os.path.join(ROOT, "tests", "cpp", "field_limits_test.cpp"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "field limits ok" in r.stdout, r.stdout + r.stderr
