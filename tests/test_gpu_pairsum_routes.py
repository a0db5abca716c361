"""Pair sums of histograms on both sides of the rules that choose their kernel: short
histograms (384 bins) bin by bin, few and many q and histograms (work groups of 256 q),
histograms over the nodes in groups as long as 14 of them need, of 1,024 bins, and, where
the products are the larger part, as long as q allows; 8 and 9 histograms.

The bar is that of tests/test_gpu_nodesum.py, per term of the sum against the oracle."""
import numpy as np
import pytest

import xansons_hip as xh
import xs_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,nhist,bin_,q1,nq", [
    (1, 383, 0.01, 20.0, 1), (1, 384, 0.01, 20.0, 300), (1, 385, 0.01, 20.0, 300),
    (4, 384, 0.3, 20.0, 65000), (4, 384, 0.3, 20.0, 66000), (1025, 20, 0.02, 10.0, 3),
    (8, 14 * 97, 0.001, 1.0, 50), (9, 14 * 97 + 1, 0.001, 1.0, 50), (1, 14 * 1024 + 1, 0.001, 1.0, 70),
    (3, 20000, 0.001, 3.0, 40), (9, 9000, 0.001, 3.0, 14563), (9, 9000, 0.001, 3.0, 14564)])
def test_routes(rows, nhist, bin_, q1, nq):
    rng = np.random.default_rng(rows * 7919 + nhist)
    h = rng.integers(0, 1000, (rows, nhist)).astype(np.uint64)
    q = np.linspace(0.3, q1, nq)
    print(f"routes: {rows} x {nhist} bins of {bin_}, {nq} q to {q1}", flush=True)
    with xh.Context(0) as ctx:
        S = ctx.hist_pairsum(h, bin_, q)
    pick = np.unique(np.linspace(0, nq - 1, 40).astype(int))
    rowp = np.unique(np.linspace(0, rows - 1, 12).astype(int))
    ref = O.hist_pairsum(h[rowp], bin_, q[pick])
    x = q[pick][:, None] * ((np.arange(nhist) + 0.5) * bin_)[None, :]
    w = 2e-15 + 2e-14 / (1 + x) + (1e-8 / x) ** 2 / np.maximum(x, 1.0)
    tol = h[rowp].astype(np.float64) @ w.T
    d = np.abs(S[np.ix_(rowp, pick)] - ref)
    assert np.all(d <= tol), float((d / tol).max())
