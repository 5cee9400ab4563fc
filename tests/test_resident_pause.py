"""The pause of the one-launch solves after time-outs (CPU).

16 solves are left to the other kernels after the first time-out, 80, 336 and then
1360 after the next ones, each counted once, and as many solves without a time-out as
the last pause was long start the row again (tests/resident_pause_check.cpp).
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_pause_after_time_outs(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "monoalg3d_c_amd", "csrc"),
                    os.path.join(ROOT, "tests", "resident_pause_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout
