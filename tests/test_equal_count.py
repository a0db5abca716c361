"""The equal-count partition of few atoms over many bins (no GPU): no more columns
than the device's tables hold, and the tiles that the window's width asks for.  The
check is C++ (tests/cpp/) compiled with g++ against the library's own header."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "softx-d-16-00083_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_columns_of_sparse_structures(tmp_path):
    exe = tmp_path / "equal_count_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-I", CSRC,
                    os.path.join(HERE, "cpp", "equal_count_check.cpp"), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.strip().endswith("ok")
