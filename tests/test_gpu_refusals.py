"""Device memory that a call can do without, refused: direct Debye sums without the
moments' slabs, pair sums and batch runs without the nodes' tables, 2D intensities
without the amplitudes give the results that they give with it.  In a process of its
own, where a hipMalloc with a limit stands before the runtime's."""
import os
import shutil
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_refused_memory(tmp_path):
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    so = tmp_path / "librefuse_alloc.so"
    subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC", os.path.join(HERE, "cpp", "refuse_alloc.cpp"),
                    "-o", str(so), "-Wl,--no-as-needed", f"-L{rocm}/lib", "-lamdhip64", f"-Wl,-rpath,{rocm}/lib",
                    "-ldl"], check=True)
    print("refused memory", flush=True)
    r = subprocess.run([sys.executable, "-u", os.path.join(HERE, "refusals_child.py"), str(so)],
                       capture_output=True, text=True, timeout=100)
    print(r.stdout + r.stderr, flush=True)
    assert r.returncode == 0 and "REFUSALS OK" in r.stdout
