"""Run by tests/test_gpu_refusals.py in a process of its own: calls whose optional device
memory is refused, against the same calls with it.  argv: the library of refuse_alloc.cpp."""
import ctypes as C
import os
import sys

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "..", "softx-d-16-00083_amd"))
shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
shim.refuse_above.argtypes = [C.c_size_t]

import xansons_hip as xh  # noqa: E402
from xansons_hip import structures as st  # noqa: E402

LIMIT, NONE = 2 << 20, C.c_size_t(-1).value


def both(name, call, bar):
    """call(ctx) with all memory and with requests above LIMIT refused."""
    print(name, flush=True)
    with xh.Context(0) as ctx:
        shim.refuse_above(NONE)
        ref = call(ctx)
    with xh.Context(0) as ctx:
        shim.refuse_above(LIMIT)
        got = call(ctx)
        n = shim.refused()
        shim.refuse_above(NONE)
    err = float(np.abs(got - ref).max() / np.abs(ref).max())
    print(f"  {n} refused, {err:.1e}", flush=True)
    assert n >= 1 and err <= bar


rng = np.random.default_rng(1)
x = rng.uniform(0, 30.0, (3, 1500))
q = st.q_mesh(0.5, 12.0, 400)
both("moments", lambda c: c.debye_pairsum(x, [900, 600], q), 1e-12)

h = rng.integers(0, 1000, (10, 3000)).astype(np.uint64)
both("nodes", lambda c: c.hist_pairsum(h, 0.01, q), 1e-12)

rot = st.uniform_rotations(8)
qv = rng.uniform(-2, 2, (20000, 3))
ff = rng.uniform(1, 2, (2, 20000))
both("amplitudes, list", lambda c: c.amp2d(x, [900, 600], qv, rot, ff), 1e-12)
both("amplitudes, grid", lambda c: c.amp2d_grid(x, [900, 600], [-2, -2, 0], [0.02, 0, 0], [0, 0.02, 0], 200, 100,
                                                rot, ff), 1e-12)

ens = st.particle_ensemble(4, seed=2, nmin=200, nmax=900)


def batch(c, graph):
    b = xh.Batch(c, [(e.xyz64(), e.el_count) for e in ens], 0.01)
    assert max(b.nhist) > 384
    out = []
    for nq in (50, 50, 60):  # (the second run asks for nothing again)
        n = shim.refused()
        out.append(b.run(q=st.q_mesh(0.5, 12.0, nq), graph=graph)[1])
        if len(out) == 2:
            assert shim.refused() == n
    b.close()
    return np.concatenate(out)


for graph in (False, True):
    both(f"batch, graph={graph}", lambda c: batch(c, graph), 1e-11)

print("batch without any", flush=True)
with xh.Context(0) as ctx:
    b = xh.Batch(ctx, [(e.xyz64(), e.el_count) for e in ens], 0.01)
    shim.refuse_above(1000)
    try:
        b.run(q=q)
        raise SystemExit("not refused")
    except xh.XSError as e:
        assert e.code == -4 or "allocation" in str(e), e
    shim.refuse_above(NONE)
    S = b.run(q=q)[1]
    assert np.isfinite(S).all() and S.any()
    b.close()
print("REFUSALS OK", flush=True)
