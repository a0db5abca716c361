"""The matrix-core pair sums' slices and the column groups of a call of its own (no GPU).
The checks are C++ (tests/cpp/) compiled with g++ against the library's own header."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "softx-d-16-00083_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_top_slices_and_wide_groups(tmp_path):
    exe = tmp_path / "mfma_slices_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-I", CSRC,
                    os.path.join(HERE, "cpp", "mfma_slices_check.cpp"), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.strip().endswith("ok")
