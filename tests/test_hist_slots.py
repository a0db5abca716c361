"""The FP64 histogram kernel's blocks of 16 x 16 atoms: the slot form of its
fixed-point floor on the CPU (tests/cpp/fixslot_check.cpp), and on the GPU the
sizes where blocks, tiles and shares of tiles end, against the oracle, bit for
bit."""
import os
import shutil
import subprocess

import numpy as np
import pytest
try:
    import torch  # noqa: F401  (first import can take a minute on a fresh box)
except ImportError:
    torch = None

import xs_oracle as O

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "softx-d-16-00083_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_slot_floor_worst_rsq(tmp_path):
    exe = tmp_path / "fixslot_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-I", CSRC,
                    os.path.join(HERE, "cpp", "fixslot_check.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("counts", [[15], [16], [17], [255, 1], [257, 240], [1008, 1009], [2047],
                                    [2064, 31], [3073, 1, 16]])
@pytest.mark.parametrize("bin_,cut,lattice", [(0.01, 1.0, False), (0.0007, 1.0, False),
                                              (0.01, 0.4, False), (0.125, 1.0, True)])
def test_block_edges(ctx, counts, bin_, cut, lattice):
    """Histograms in the 8,192-bin window, beyond the 32,768-bin one, cut below
    the largest distance, and with distances on bin edges (a lattice of 1/4 A,
    some atoms on the same site)."""
    n = sum(counts)
    rng = np.random.default_rng(n)
    x = rng.uniform(0, 18.0, (3, n))
    if lattice:
        x = np.round(x * 4) / 4
    nh = max(1, int(O.hist_size(x, bin_) * cut))
    print(f"blocks {counts} bin {bin_} nhist {nh}", flush=True)
    h, ov = ctx.hist(x, counts, bin_, nh, f64=True)
    ho, oo = O.hist_f64(x, counts, bin_, nh)
    assert ov == oo
    assert np.array_equal(h, ho)
