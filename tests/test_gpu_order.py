"""Histograms whose atoms the device puts into equal-count tiles, at the sizes and
shapes where that can go wrong: elements of no atom, one and around a tile of 1,024,
flat structures, all atoms at one point, planes of a lattice, two clusters far apart,
and ensembles of such structures.  Counts are compared with the oracle's bit for bit."""
import numpy as np
import pytest
try:
    import torch  # noqa: F401  (first import can take a minute on a fresh box)
except ImportError:
    torch = None

import xansons_hip as xh
import xs_oracle as O

pytestmark = pytest.mark.gpu
BIN = 0.02


def shape(kind, n, seed=1):
    rng = np.random.default_rng(seed + n)
    x = rng.uniform(-12.0, 12.0, (3, n))
    if kind == "flat":
        x[0] = 1.5
    elif kind == "line":
        x[:2] = [[0.25], [-3.0]]
    elif kind == "point":
        x[:] = 2.0
    elif kind == "lattice":
        x = np.round(x / 4.0) * 4.0
    elif kind == "clusters":
        x = x * 0.05 + np.where(rng.uniform(size=n) < 0.5, -40.0, 40.0)
    return np.ascontiguousarray(x)


CASES = [("box", [1]), ("box", [0, 2, 0]), ("box", [31, 33]), ("box", [1023]), ("box", [1024, 1]),
         ("box", [1025, 2049, 64]), ("flat", [3000]), ("line", [2500, 100]), ("point", [1500]),
         ("lattice", [4000, 700]), ("clusters", [5000])]


@pytest.fixture(scope="module")
def ctx():
    with xh.Context(0) as c:
        yield c


@pytest.mark.parametrize("kind,counts", CASES)
@pytest.mark.parametrize("f64", [True, False])
def test_order(ctx, kind, counts, f64):
    x = shape(kind, sum(counts))
    nh = O.hist_size(x, BIN) + 2
    print(f"order: {kind} {counts} f64 {f64} {nh} bins", flush=True)
    if f64:
        got, ovf = ctx.hist(x, counts, BIN, nh, f64=True)
        want, _ = O.hist_f64(x, counts, BIN, nh)
    else:
        x = x.astype(np.float32)
        got, ovf = ctx.hist(x, counts, BIN, nh)
        want, _ = O.hist_f32(x, counts, BIN, nh)
    assert ovf == 0
    assert np.array_equal(got, want)


@pytest.mark.parametrize("f64", [True, False])
def test_order_of_an_ensemble(ctx, f64):
    xs = [shape(k, sum(c)) for k, c in CASES]
    dev = [torch.from_numpy(x).cuda() for x in xs]
    nh = [O.hist_size(x, BIN) + 2 for x in xs]
    torch.cuda.synchronize()
    print(f"order: ensemble f64 {f64}", flush=True)
    b = xh.Batch(ctx, [(d.data_ptr(), c) for d, (_, c) in zip(dev, CASES)], BIN, nhist=nh, f64=f64, device=True)
    hist = np.concatenate([np.asarray(h).ravel() for h in b.run()[0]])
    b.close()
    o = 0
    for x, (_, c), h in zip(xs, CASES, nh):
        nt = len(c) * (len(c) + 1) // 2
        want = (O.hist_f64(x, c, BIN, h) if f64 else O.hist_f32(x.astype(np.float32), c, BIN, h))[0]
        assert np.array_equal(hist[o:o + nt * h].reshape(nt, h), want)
        o += nt * h
