"""2D intensities at the sizes where the kernels can go wrong.  Regular q grid: rows of 1, 15, 16, 17 and more points, one row, atoms around a step of 4 and a
chunk of 128, empty elements, few runs (the atoms in shares), many (one share) and
very many (two tiles a wave).  List: atoms
around a chunk of 256, points around a block, shares.  Both under stream capture.

The bar: a term's seed is a hardware sine of an FP32 phase, 2^-25 turn and 2^-22, so
each of its parts is within 5e-7 and an amplitude within a = 5e-7 sqrt(2) sum f n;
|A|^2 then moves by at most 2 |A| a + a^2."""
import numpy as np
import pytest
try:
    import torch  # noqa: F401  (first import can take a minute on a fresh box)
except ImportError:
    torch = None

import xansons_hip as xh
from xansons_hip import structures as st

pytestmark = pytest.mark.gpu


def reference(x, counts, q, rot, ff):
    off = np.concatenate([[0], np.cumsum(counts)])
    ref, bar = np.zeros(len(q)), np.zeros(len(q))
    for R in rot:
        A, a = np.zeros(len(q), complex), np.zeros(len(q))
        y = R @ x  # (R^T q).x = q.(R x)
        for e, c in enumerate(counts):
            for k in range(0, len(q), 4096):
                A[k:k + 4096] += ff[e, k:k + 4096] * np.exp(
                    1j * (q[k:k + 4096] @ y[:, off[e]:off[e + 1]])).sum(axis=1)
            a += 5e-7 * np.sqrt(2.0) * c * ff[e]
        ref += np.abs(A) ** 2
        bar += 2 * np.abs(A) * a + a * a
    return ref, bar


@pytest.mark.parametrize("counts,nu,nv,nrot", [
    ([1], 1, 1, 1), ([3], 16, 1, 1), ([4, 5], 17, 3, 2), ([127, 1, 130], 33, 9, 2),
    ([128], 15, 70, 3), ([0, 129, 300], 48, 5, 1), ([2000, 1], 31, 40, 2),
    ([700], 40, 1100, 4), ([3, 2], 33, 65500, 1)])
def test_amp2d_grid_edges(counts, nu, nv, nrot):
    n = sum(counts)
    rng = np.random.default_rng(n + nu)
    x = rng.uniform(-40.0, 40.0, (3, n))
    q0, du, dv = np.array([-3.0, 2.0, 0.3]), np.array([0.11, 0.02, 0.0]), np.array([-1e-3, 0.013, 0.004])
    rot = st.uniform_rotations(nrot, seed=2).reshape(-1, 3, 3)
    ff = rng.uniform(0.5, 2.0, (len(counts), nu * nv))
    print(f"grid: {counts} atoms, {nu} x {nv} points, {nrot} rotations", flush=True)
    with xh.Context(0) as ctx:
        I = ctx.amp2d_grid(x, counts, q0, du, dv, nu, nv, rot.reshape(-1, 9), ff)
    v3 = np.arange(nv)[:, None, None] * dv + np.arange(nu)[None, :, None] * du + q0
    ref, bar = reference(x, counts, v3.reshape(-1, 3), rot, ff)
    assert np.all(np.abs(I - ref) <= bar + 1e-12 * ref.max())


@pytest.mark.parametrize("counts,npts,nrot", [
    ([1], 1, 1), ([255, 256, 257], 255, 2), ([0, 1025], 256, 3), ([700, 900], 257, 2), ([300], 70000, 8)])
def test_amp2d_list_edges(counts, npts, nrot):
    n = sum(counts)
    rng = np.random.default_rng(n + npts)
    x, q = rng.uniform(-40.0, 40.0, (3, n)), rng.uniform(-4.0, 4.0, (npts, 3))
    rot = st.uniform_rotations(nrot, seed=2).reshape(-1, 3, 3)
    ff = rng.uniform(0.5, 2.0, (len(counts), npts))
    print(f"list: {counts} atoms, {npts} points, {nrot} rotations", flush=True)
    with xh.Context(0) as ctx:
        I = ctx.amp2d(x, counts, q, rot.reshape(-1, 9), ff)
    ref, bar = reference(x, counts, q, rot, ff)
    assert np.all(np.abs(I - ref) <= bar + 1e-12 * ref.max())


@pytest.mark.parametrize("grid", [False, True])
def test_amp2d_stream_capture(grid):
    """A captured call keeps no pointer to the context's scratch."""
    rng = np.random.default_rng(4)
    n, nu, nv = 3000, 20, 16
    rot = st.uniform_rotations(2, seed=2).reshape(-1, 9)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    xd, qd, rd = dev(rng.uniform(-30, 30, (3, n))), dev(rng.uniform(-3, 3, (nu * nv, 3))), dev(rot)
    fd, I = dev(rng.uniform(0.5, 2.0, (1, nu * nv))), torch.empty(nu * nv, dtype=torch.float64, device="cuda")
    big = rng.uniform(-1, 1, (20000, 3))
    with xh.Context(0) as c:
        def run():
            if grid:
                c.amp2d_grid_dev(xd.data_ptr(), n, [n], [-2.0, 1.0, 0.0], [0.1, 0.0, 0.0], [0.0, 0.1, 0.01],
                                 nu, nv, rd.data_ptr(), 2, fd.data_ptr(), I.data_ptr())
            else:
                c.amp2d_dev(xd.data_ptr(), n, [n], qd.data_ptr(), nu * nv, rd.data_ptr(), 2, fd.data_ptr(),
                            I.data_ptr())
        stream = torch.cuda.Stream()
        torch.cuda.synchronize()
        c.set_stream(stream.cuda_stream)
        run()
        c.synchronize()
        ref = I.cpu().numpy()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=stream):
            run()
        for k in range(3):
            c.amp2d(big.T[:, :1100], [1100], big[:(k + 1) * 6000], rot, np.ones((1, (k + 1) * 6000)))
            I.fill_(7.0)
            torch.cuda.synchronize()
            with torch.cuda.stream(stream):
                g.replay()
            torch.cuda.synchronize()
            assert np.abs(I.cpu().numpy() - ref).max() <= 1e-12 * ref.max()
        c.set_stream(0)
