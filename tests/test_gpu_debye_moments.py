"""The direct Debye sums through Chebyshev moments at the sizes where they can
go wrong: segments of 1, 63, 64 and 65 atoms, atoms that coincide or almost do
(the bin that reaches r = 0), q ranges that take few and many moments, blocks,
uniform and other meshes.

Bars, per pair type and relative to max |S|.  On any mesh against the
allocation-free entry point (32 x 32 tiles, every pair against every q): 1e-12,
the bar of its own tests.  On a mesh that is not uniform also against the
oracle: truncation 5e-13 a pair with varying sign and the second order of the
denominator's 1e-8 leave 1e-11."""
import numpy as np
import pytest
try:
    import torch  # noqa: F401  (first import can take a minute on a fresh box)
except ImportError:
    torch = None

import xansons_hip as xh
import xs_oracle as O
from xansons_hip import structures as st

pytestmark = pytest.mark.gpu


def atoms(counts, box, seed, near=0, same=0):
    """Uniform atoms in a box; the last `near` are moved next to the first ones
    (1e-3 A), the last `same` before them onto them."""
    rng = np.random.default_rng(seed)
    n = sum(counts)
    x = rng.uniform(-box / 2, box / 2, (3, n))
    if near:
        x[:, n - near:] = x[:, :near] + 1e-3 * rng.uniform(-1, 1, (3, near))
    if same:
        x[:, n - near - same:n - near] = x[:, :same]
    return np.ascontiguousarray(x)


def scaled(a, b):
    s = np.maximum(np.abs(b).max(axis=-1, keepdims=True), 1e-300)
    return float((np.abs(a - b) / s).max())


@pytest.mark.parametrize("counts,box,q,near,same", [
    ([1500], 30.0, (0.5, 6.0, 400), 0, 0),
    ([1, 1345, 63, 64, 65], 40.0, (0.3, 10.0, 1024), 0, 0),
    ([1281, 700], 25.0, (0.0, 12.0, 777), 9, 5),
    ([2000, 513], 120.0, (0.2, 25.0, 1000), 3, 0),
    ([3000], 300.0, (0.2, 20.0, 1500), 0, 2),
])
def test_uniform_mesh(counts, box, q, near, same):
    x = atoms(counts, box, 7, near, same)
    qm = st.q_mesh(*q)
    with xh.Context(0) as ctx:
        xd, qd = torch.from_numpy(x).cuda(), torch.from_numpy(qm).cuda()
        P = len(counts) * (len(counts) + 1) // 2
        a, b = (torch.full((P, qm.size), 5.0, dtype=torch.float64, device="cuda") for _ in range(2))
        torch.cuda.synchronize()
        print(f"moments: {counts} box {box} q {q}", flush=True)
        ctx.debye_pairsum_dev(xd.data_ptr(), x.shape[1], counts, qd.data_ptr(), qm.size, a.data_ptr())
        ctx.debye_pairsum_noalloc_dev(xd.data_ptr(), x.shape[1], counts, qd.data_ptr(), qm.size,
                                      b.data_ptr())
        ctx.synchronize()
        err = scaled(a.cpu().numpy(), b.cpu().numpy())
    print(f"  {err:.2e}", flush=True)
    assert err <= 1e-12


@pytest.mark.parametrize("counts,blocks", [([1500, 321], 1), ([1200, 900], 3)])
def test_other_mesh_and_blocks(counts, blocks):
    x = atoms(counts, 35.0, 11)
    rng = np.random.default_rng(5)
    q = np.sort(rng.uniform(0.3, 14.0, 300))
    blk = np.concatenate([rng.multinomial(c, [1.0 / blocks] * blocks) for c in counts])
    with xh.Context(0) as ctx:
        if blocks == 1:
            S = ctx.debye_pairsum(x, counts, q)
            ref = O.debye_pairsum(x, counts, q)
        else:
            S = ctx.partial_debye_pairsum(x, counts, blk, blocks, q)
            ref = O.partial_debye_pairsum(x, counts, blk, blocks, q)
    err = scaled(S, np.asarray(ref).reshape(S.shape))
    print(f"moments {counts}, {blocks} blocks: {err:.2e}", flush=True)
    assert err <= 1e-11
