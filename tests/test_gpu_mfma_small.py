"""Small calls on the int8 matrix cores, on both sides of the rules that they change:
columns in one launch whatever their slices (below 16 k tiles a CU) or in waves side by
side, tables as arguments (128 columns) or copied, extents by one work group a column
(4,096 bins) or several, the top slice left out from 17 k tiles on.

The bar is that of tests/test_gpu_mfma_edges.py."""
import numpy as np
import pytest

import xansons_hip as xh
import xs_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncols,nhist,nq", [
    (1, 1, 1), (9, 50, 2000), (100, 100, 1500), (128, 64, 40), (129, 64, 40), (3, 511, 300), (3, 513, 300),
    (2, 4096, 130), (2, 4097, 130), (70, 5000, 3300), (70, 5100, 3400)])
def test_small(ncols, nhist, nq):
    rng = np.random.default_rng(ncols + nhist)
    bits = rng.integers(0, 35, ncols)
    h = np.stack([rng.integers(0, 1 << b, nhist) if b else np.zeros(nhist, np.int64) for b in bits]).astype(np.uint64)
    h[:, nhist * 2 // 3:][::2] = 0  # columns that end early
    q = np.linspace(0.4, 25.0, nq)
    print(f"mfma small: {ncols} x {nhist} bins, {nq} q", flush=True)
    with xh.Context(0) as ctx:
        S = ctx.hist_pairsum(h, 0.02, q, mfma=True)
    pick = np.unique(np.linspace(0, nq - 1, 60).astype(int))
    ref = O.hist_pairsum(h, 0.02, q[pick])
    bar = (2.0 ** -35 + 1e-13) * h.astype(np.float64).sum(axis=1, keepdims=True)
    assert np.all(np.abs(S[:, pick] - ref) <= bar)


def test_huge_q():
    """|q| r beyond 1e77, where the product of four denominators would overflow: terms of 0,
    and the other q as without them."""
    h = np.arange(1, 301, dtype=np.uint64).reshape(2, 150)
    q = np.array([0.5, 1e78, 2.0, -1e90, 1e200, 3.0])
    print("mfma: huge q", flush=True)
    with xh.Context(0) as ctx:
        S = ctx.hist_pairsum(h, 0.02, q, mfma=True)
    small = np.abs(q) < 10
    bar = (2.0 ** -35 + 1e-13) * h.astype(np.float64).sum(axis=1, keepdims=True)
    assert np.all(np.abs(S[:, small] - O.hist_pairsum(h, 0.02, q[small])) <= bar)
    assert np.all(np.abs(S[:, ~small]) <= bar)
