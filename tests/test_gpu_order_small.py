"""Histograms of few atoms, whose ordering takes one work group: around its limit of 4,096
atoms, 16 elements, a lattice, columns too many for its counters (the last one), and a
small ensemble.  Counts are compared with the oracle's bit for bit."""
import numpy as np
import pytest
try:
    import torch  # noqa: F401  (first import can take a minute on a fresh box)
except ImportError:
    torch = None

import xansons_hip as xh
import xs_oracle as O

pytestmark = pytest.mark.gpu


def atoms(n, grid, seed=3):
    x = np.random.default_rng(seed + n).uniform(-12.0, 12.0, (3, n))
    return np.ascontiguousarray(np.round(x / grid) * grid if grid else x)


def want(x, counts, b, nh, f64):
    return (O.hist_f64(x, counts, b, nh) if f64 else O.hist_f32(x.astype(np.float32), counts, b, nh))[0]


@pytest.mark.parametrize("f64", [True, False])
@pytest.mark.parametrize("counts,b,grid", [
    ([4095], 0.02, 0), ([4096], 0.02, 0), ([4097], 0.02, 0), ([1, 2047, 2048], 0.02, 0),
    ([200] * 16, 0.02, 0), ([3000, 900], 0.02, 4.0), ([1500, 2500], 1e-3, 0), ([4000], 2e-4, 0)])
def test_small(counts, b, grid, f64):
    x = atoms(sum(counts), grid)
    nh = O.hist_size(x, b) + 2
    print(f"order: {counts} atoms, f64 {f64}, {nh} bins", flush=True)
    with xh.Context(0) as ctx:
        got, ovf = ctx.hist(x if f64 else x.astype(np.float32), counts, b, nh, f64=f64)
    assert ovf == 0
    assert np.array_equal(got, want(x, counts, b, nh, f64))


@pytest.mark.parametrize("f64", [True, False])
def test_small_ensemble(f64):
    parts = [[300, 0, 5], [1], [0, 1700], [2000]]
    xs = [atoms(sum(c), 0, seed=i) for i, c in enumerate(parts)]
    dev = [torch.from_numpy(x).cuda() for x in xs]
    nh = [O.hist_size(x, 0.02) + 2 for x in xs]
    torch.cuda.synchronize()
    print(f"order: small ensemble, f64 {f64}", flush=True)
    with xh.Context(0) as ctx:
        p = xh.Batch(ctx, [(d.data_ptr(), c) for d, c in zip(dev, parts)], 0.02, nhist=nh, f64=f64, device=True)
        hist = np.concatenate([np.asarray(h).ravel() for h in p.run()[0]])
        p.close()
    assert np.array_equal(hist, np.concatenate(
        [want(x, c, 0.02, h, f64).ravel() for x, c, h in zip(xs, parts, nh)]))
