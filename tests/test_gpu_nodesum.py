"""Pair sums of histograms over Chebyshev nodes at the sizes where they can go
wrong: one histogram, the last few that take the product with groups as rows and
the first that take the product with histograms as rows (8, 9), tiles of 16;
histograms that end at a group of bins or one beyond it, 16 groups and 17; every
bin a node; groups of the largest size; q = 0 and negative q; partly filled blocks
of q; more groups than one pass holds.

The bar, per term of the sum against the oracle: the phase q r is rounded in both
(2e-15 of the count), sines, interpolation and weights 2e-14 of the count times
1/(1 + q r), and the second order of the denominator's 1e-8, (1e-8/(q r))^2."""
import numpy as np
import pytest
try:
    import torch  # noqa: F401  (first import can take a minute on a fresh box)
except ImportError:
    torch = None

import xansons_hip as xh
import xs_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with xh.Context(0) as c:
        yield c


def check(ctx, rows, nhist, bin_, q):
    rng = np.random.default_rng(rows * 7919 + nhist)
    h = rng.integers(0, 1000, (rows, nhist)).astype(np.uint64)
    q = np.asarray(q, np.float64)
    print(f"nodes: {rows} x {nhist} bins of {bin_}, {q.size} q to {np.abs(q).max()}", flush=True)
    S = ctx.hist_pairsum(h, bin_, q)
    ref = O.hist_pairsum(h, bin_, q)
    x = np.abs(q)[:, None] * ((np.arange(nhist) + 0.5) * bin_)[None, :]
    with np.errstate(divide="ignore"):
        w = 2e-15 + 2e-14 / (1 + x) + np.where(x > 0, (1e-8 / x) ** 2, 0.0) / np.maximum(x, 1.0)
    tol = h.astype(np.float64) @ w.T
    assert np.all(S[:, q == 0] == 0.0)
    assert np.all(np.abs(S - ref) <= tol), float((np.abs(S - ref) / np.maximum(tol, 1e-300)).max())


# 0.01 A and 20 1/A: 284 bins a group
@pytest.mark.parametrize("rows,nhist", [
    (1, 1), (1, 63), (2, 283), (3, 284), (8, 285), (9, 285), (16, 569), (17, 1000),
    (1, 14 * 284), (2, 14 * 284 + 1), (8, 15 * 284 + 1), (9, 16 * 284 + 1), (33, 3000), (130, 700)])
@pytest.mark.parametrize("nq", [1, 65])
def test_groups(ctx, rows, nhist, nq):
    check(ctx, rows, nhist, 0.01, np.linspace(0.3, 20.0, nq) if nq > 1 else [20.0])


@pytest.mark.parametrize("rows,nhist,bin_,q", [
    (1, 64, 0.2, (0.5, 30.0, 16)),        # every bin a node
    (3, 1025, 0.2, (0.5, 30.0, 17)),
    (8, 65, 0.2, (0.5, 30.0, 64)),
    (20, 777, 0.2, (0.5, 30.0, 64)),
    (2, 9000, 1e-4, (0.5, 1.0, 40)),      # 4,096 bins a group
    (12, 9000, 1e-4, (0.5, 1.0, 40)),
    (1, 300, 0.05, (0.4, 11.0, 16385)),   # the plan by a kernel of its own
    (2, 64 * 32768 + 3, 0.01, (50.0, 100.0, 3)),  # two passes over the groups
    (9, 64 * 32768 + 3, 0.01, (50.0, 100.0, 3)),
])
def test_forms(ctx, rows, nhist, bin_, q):
    check(ctx, rows, nhist, bin_, np.linspace(*q))


@pytest.mark.parametrize("rows", [2, 11])
def test_zero_and_negative_q(ctx, rows):
    check(ctx, rows, 1500, 0.01, [0.0, -3.0, 7.5, -20.0, 0.0, 0.4])
    S = ctx.hist_pairsum(np.ones((rows, 50), np.uint64), 0.1, np.zeros(3))
    assert np.all(S == 0.0)


def test_stream_capture(ctx):
    """A captured call keeps no pointer to the context's scratch: replayed after a
    larger call has moved it, and between eager calls."""
    rng = np.random.default_rng(3)
    q = np.linspace(0.3, 20.0, 300)
    h = rng.integers(0, 1000, (3, 5000)).astype(np.uint64)
    ref = O.hist_pairsum(h, 0.01, q)
    bar = 1e-12 * np.abs(ref).max()
    with xh.Context(0) as c:
        hd, qd = torch.from_numpy(h.astype(np.int64)).cuda(), torch.from_numpy(q).cuda()
        S = torch.empty((3, q.size), dtype=torch.float64, device="cuda")
        run = lambda: c.hist_pairsum_dev(hd.data_ptr(), 3, 5000, 0.01, qd.data_ptr(), q.size, S.data_ptr())
        stream = torch.cuda.Stream()
        torch.cuda.synchronize()
        c.set_stream(stream.cuda_stream)
        run()
        c.synchronize()
        assert np.abs(S.cpu().numpy() - ref).max() <= bar
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=stream):
            run()
        for k in range(3):
            c.hist_pairsum(np.ones((40 * (k + 1), 9000 * (k + 1)), np.uint64), 0.01, q)
            S.fill_(7.0)
            torch.cuda.synchronize()
            with torch.cuda.stream(stream):
                g.replay()
            torch.cuda.synchronize()
            assert np.abs(S.cpu().numpy() - ref).max() <= bar
        c.set_stream(0)
