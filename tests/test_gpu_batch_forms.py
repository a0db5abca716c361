"""One batch plan run in one form and then in another: pair sums on the matrix
cores, over the nodes and on the matrix cores again, with another nq or other
outputs in between, eager and as graph replays.  Every run's pair sums against
the oracle: 1e-9 of max |S| on the matrix cores (the bar of their own tests),
1e-11 over the nodes."""
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

BIN = 0.02
Q = st.q_mesh(0.4, 15.0, 200)
Q2 = st.q_mesh(0.3, 9.0, 333)


@pytest.fixture(scope="module")
def ens():
    return [st.random_cluster([90, 60], box=11.0, min_dist=0.8, seed=s) for s in (1, 2)] + \
        [st.random_cluster([150], box=9.0, min_dist=0.7, seed=3)]


def oracle(b, hist, q):
    rows = []
    for s in range(len(b.nhist)):
        h0, nh = int(b.hist_off[s]), int(b.nhist[s])
        h1 = int(b.hist_off[s + 1]) if s + 1 < len(b.nhist) else b.hist_len
        rows.append(O.hist_pairsum(hist[h0:h1].reshape(-1, nh), BIN, q))
    return np.concatenate(rows)


def check(S, ref, mfma, label):
    err = float((np.abs(S.reshape(ref.shape) - ref) / np.abs(ref).max(axis=1, keepdims=True)).max())
    print(f"{label}: {err:.2e}", flush=True)
    assert err <= (1e-9 if mfma else 1e-11)


def test_host_runs_of_every_form(ens):
    """(mfma, q, with PDF): a run with PDFs stages more than one without."""
    with xh.Context(0) as ctx:
        b = xh.Batch(ctx, [(e.xyz64(), e.el_count) for e in ens], BIN)
        sl, rho = np.full(sum(e.n_el for e in ens), 3.0), np.full(len(ens), 0.05)
        ref = None
        for mfma, q, pdf in [(True, Q, False), (False, Q, False), (True, Q, False), (False, Q, True),
                             (True, Q, False), (True, Q2, True), (False, Q2, False), (True, Q2, True),
                             (True, Q, True)]:
            print(f"host mfma={mfma} nq={q.size} pdf={pdf}", flush=True)
            kw = dict(pdf_type="rPDF", rho0=rho, sl=sl) if pdf else {}
            hist, S, _ = b.run(q=q, mfma=mfma, **kw)
            if ref is None:
                ref = {x.size: oracle(b, hist, x) for x in (Q, Q2)}
            check(S, ref[q.size], mfma, "  S")
        b.close()


@pytest.mark.parametrize("graph", [False, True])
def test_device_runs_of_every_form(ens, graph):
    """On device arrays, whose runs stage nothing: the nodes' tables of one run
    follow the kept regions directly, as the matrix-core slices of another do."""
    with xh.Context(0) as ctx:
        b = xh.Batch(ctx, [(e.xyz64(), e.el_count) for e in ens], BIN)
        hist = torch.empty(b.hist_len, dtype=torch.int64, device="cuda")
        ref = None
        for n, (mfma, q) in enumerate([(True, Q), (False, Q), (True, Q), (True, Q), (False, Q2),
                                       (True, Q2), (True, Q), (False, Q), (True, Q)]):
            qd = torch.from_numpy(q).cuda()
            S = torch.full((b.ntypes_total * q.size,), float("nan"), dtype=torch.float64, device="cuda")
            torch.cuda.synchronize()
            print(f"device mfma={mfma} nq={q.size} graph={graph and not (n & 1)}", flush=True)
            # (graph: every other run eager, between the replays)
            b.run_dev(hist.data_ptr(), qd.data_ptr(), q.size, S.data_ptr(), mfma=mfma,
                      graph=graph and not (n & 1))
            ctx.synchronize()
            if ref is None:
                h = hist.cpu().numpy().view(np.uint64)
                ref = {x.size: oracle(b, h, x) for x in (Q, Q2)}
            check(S.cpu().numpy(), ref[q.size], mfma, "  S")
        b.close()


def test_graph_replays_after_an_eager_run_of_another_form(ens):
    """One captured matrix-core graph, replayed on the same buffers after an eager
    run over the nodes and after one that had to grow the buffer."""
    with xh.Context(0) as ctx:
        b = xh.Batch(ctx, [(e.xyz64(), e.el_count) for e in ens], BIN)
        hist = torch.empty(b.hist_len, dtype=torch.int64, device="cuda")
        qd, S, S2 = torch.from_numpy(Q).cuda(), *(torch.empty(b.ntypes_total * Q.size, dtype=torch.float64,
                                                             device="cuda") for _ in range(2))
        torch.cuda.synchronize()
        ref = None
        for rep in range(3):
            print(f"replay {rep}", flush=True)
            S.fill_(float("nan"))
            torch.cuda.synchronize()
            b.run_dev(hist.data_ptr(), qd.data_ptr(), Q.size, S.data_ptr(), mfma=True, graph=True)
            ctx.synchronize()
            if ref is None:
                ref = oracle(b, hist.cpu().numpy().view(np.uint64), Q)
            check(S.cpu().numpy(), ref, True, "  graph")
            b.run_dev(hist.data_ptr(), qd.data_ptr(), Q.size, S2.data_ptr())
            ctx.synchronize()
            check(S2.cpu().numpy(), ref, False, "  eager")
            if rep == 1:
                b.run(q=np.resize(Q, 20000))  # a host run with much more to stage
        b.close()
