"""Rows applied from neighbourhood masks against the oracle's rows (CPU).

The solve kernels multiply by a 27-point anisotropic row without forming it:
as sums of masked differences with weights from a table of the layer
(monoalg3d_c_amd/csrc/aniso_row.h).  Built for the host, that product must
agree with the oracle's assembled rows times the same values
(oracle/assembly.c, assembly_common.c:115-830) in FP64 and FP32, on boxes with
none to half of the cells inactive, with every cross term and with one only,
and whatever inactive cells hold.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.parametrize("flags", [["-ffp-contract=off"], ["-ffp-contract=fast"]])
def test_mask_products_match_oracle_rows(tmp_path, flags):
    if not os.path.exists(HIPCC) or shutil.which("gcc") is None:
        pytest.skip("hipcc / gcc not available")
    src = os.path.join(ROOT, "tests", "mask_apply_check.cpp")
    asm_o, chk_o, exe = (str(tmp_path / n) for n in ("assembly.o", "chk.o", "chk"))
    subprocess.run(["gcc", "-O2", "-ffp-contract=off", "-c", os.path.join(ROOT, "oracle", "assembly.c"), "-o", asm_o,
                    "-I", os.path.join(ROOT, "oracle")], check=True)
    subprocess.run([HIPCC, "-O2", *flags, "-std=c++17", "-I", os.path.join(ROOT, "monoalg3d_c_amd", "csrc"),
                    "-I", os.path.join(ROOT, "include"), "-c", src, "-o", chk_o], check=True, capture_output=True)
    subprocess.run([HIPCC, chk_o, asm_o, "-o", exe], check=True, capture_output=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
    assert r.stdout.count("of the diagonal") == 8
