"""2D intensities on a regular q grid at the sizes where the kernel can go wrong:
rows of 1, 15, 16, 17 and more points, one row, atoms around a step of 4 and a
chunk of 128, empty elements, few runs (the atoms in shares), many (one share) and
very many (two tiles a wave).

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
    off = np.concatenate([[0], np.cumsum(counts)])
    ref, bar = np.zeros(nu * nv), np.zeros(nu * nv)
    for R in rot:
        A, a = np.zeros(nu * nv, complex), np.zeros(nu * nv)
        y = R @ x  # (R^T q).x = q.(R x)
        u = np.exp(1j * np.outer(np.arange(nu), du @ y))
        v = np.exp(1j * np.outer(np.arange(nv), dv @ y)) * np.exp(1j * (q0 @ y))
        for e, c in enumerate(counts):
            s = slice(off[e], off[e + 1])
            A += ff[e] * (v[:, s] @ u[:, s].T).ravel()
            a += 5e-7 * np.sqrt(2.0) * c * ff[e]
        ref += np.abs(A) ** 2
        bar += 2 * np.abs(A) * a + a * a
    assert np.all(np.abs(I - ref) <= bar + 1e-12 * ref.max())
