"""Pair sums on the int8 matrix cores at the sizes where the slices and the product can
go wrong: columns around one and two waves' tiles (32, 64, 128), q around a tile of 32
and a block of 128, bins around a k tile of 32 and the four that a thread slices, few
work groups (the k range in shares) and many, counts of one to five 7-bit slices.

The bar: the sine table is within 2^-35 of its value, so a sum is within
2^-35 sum h, and the FP64 rest within 1e-13 sum h."""
import numpy as np
import pytest
try:
    import torch  # noqa: F401  (first import can take a minute on a fresh box)
except ImportError:
    torch = None

import xansons_hip as xh
import xs_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncols,nhist,nq,bits", [
    (1, 31, 1, 7), (32, 32, 31, 7), (33, 33, 33, 14), (64, 127, 128, 14), (65, 129, 129, 7),
    (128, 640, 64, 21), (129, 4096, 257, 14), (40, 33000, 40, 28), (70, 1000, 5000, 35),
    (5, 70000, 33, 7)])
def test_mfma_edges(ncols, nhist, nq, bits):
    rng = np.random.default_rng(ncols + nhist)
    h = rng.integers(0, 1 << bits, (ncols, nhist)).astype(np.uint64)
    q = np.concatenate([[0.0], np.linspace(0.4, 25.0, nq - 1)]) if nq > 2 else np.array([3.0])
    print(f"mfma: {ncols} x {nhist} bins, {q.size} q, {bits} bits", flush=True)
    with xh.Context(0) as ctx:
        S = ctx.hist_pairsum(h, 0.004, q, mfma=True)
    ref = O.hist_pairsum(h, 0.004, q)
    bar = (2.0 ** -35 + 1e-13) * h.astype(np.float64).sum(axis=1, keepdims=True)
    assert np.all(S[:, q == 0] == 0.0)
    assert np.all(np.abs(S - ref) <= bar)
