"""The radix sort's digits over one and two ranges of a key's bits, compiled for the
host: their passes order keys as a stable sort by the ranges does, with anything in
the bits between.  Needs hipcc (the HIP headers), not a GPU."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(ROOT, "vnm-graph-reordering_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is not installed")
def test_digits_order_as_the_ranges_do(tmp_path):
    exe = str(tmp_path / "key_bits_check")
    subprocess.run([HIPCC, "-O1", "-g", "-std=c++17", "-Xarch_host", "-fsanitize=undefined",
                    "-Xarch_host", "-fno-sanitize-recover=undefined",
                    "-I" + os.path.join(ROOT, "include"), "-I" + CSRC,
                    os.path.join(HERE, "key_bits_check.cpp"), "-o", exe],
                   check=True, capture_output=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
