"""Histograms of few atoms over many bins, whose windows ask for more slabs and columns
than there are atoms: counts equal the oracle's, from host arrays and in a plan tiled
on the device."""
import numpy as np
import pytest
try:
    import torch  # noqa: F401  (first import can take a minute on a fresh box)
except ImportError:
    torch = None

import xansons_hip as xh
import xs_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts,edge,bin_", [
    ([300, 2], 500.0, 1e-4),     # 588 x 588 columns by the window
    ([40], 9000.0, 1e-4),        # 10,600 x 10,600
    ([1025, 700], 100.0, 1e-3),  # 12 x 12
])
def test_sparse_f64(counts, edge, bin_):
    rng = np.random.default_rng(len(counts))
    x = rng.uniform(0, edge, (3, sum(counts)))
    nh = O.hist_size(x, bin_)
    with xh.Context(0) as ctx:
        print(f"sparse: {counts} atoms, {nh} bins", flush=True)
        h, ovf = ctx.hist(x, counts, bin_, nh, f64=True)
    ref, ovf_ref = O.hist_f64(x, counts, bin_, nh)
    assert ovf == ovf_ref and np.array_equal(h, ref)


def test_sparse_device_plan():
    rng = np.random.default_rng(5)
    xs = [rng.uniform(0, e, (3, n)) for n, e in ((200, 300.0), (1, 1.0), (90, 3000.0))]
    with xh.Context(0) as ctx:
        d = [torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in xs]
        torch.cuda.synchronize()
        print("sparse device plan", flush=True)
        b = xh.Batch(ctx, [(t.data_ptr(), [x.shape[1]]) for t, x in zip(d, xs)], 1e-3, device=True)
        hist, _, _ = b.run()
        for s, x in enumerate(xs):
            nh = int(b.nhist[s])
            ref, _ = O.hist_f64(x, [x.shape[1]], 1e-3, nh)
            assert np.array_equal(hist[int(b.hist_off[s]):int(b.hist_off[s]) + nh], ref[0]), s
        b.close()
