"""The host side of large device-to-host copies under sanitizers, on the CPU
(tests/cpp/host_copy_test.cpp, tipl_amd/csrc/host_copy.hpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("flags", [["-fsanitize=address,undefined", "-fno-sanitize-recover=all"],
                                   ["-fsanitize=thread"]], ids=["asan", "tsan"])
def test_staged_copy(tmp_path, flags):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "host_copy_test")
    r = subprocess.run([gxx, "-std=c++17", "-O1", "-g", "-Wall", "-Wextra", *flags,
                        os.path.join(ROOT, "tests", "cpp", "host_copy_test.cpp"), "-o", exe, "-pthread"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    env = dict(os.environ, ASAN_OPTIONS="verify_asan_link_order=0")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120, env=env)
    assert r.returncode == 0 and "host copy ok" in r.stdout, r.stdout + r.stderr
