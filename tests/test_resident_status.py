"""What the host makes of the one-launch solves' record (CPU).

A solve that block 0 has counted while another block gave up in its last
exchange is not done: its step has to be solved anew.  That cannot be brought
about at will on the GPU, so the host's reading of the record is checked on
records made up for it (tests/resident_status_check.cpp).
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_record_of_solves(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "monoalg3d_c_amd", "csrc"),
                    os.path.join(ROOT, "tests", "resident_status_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout
