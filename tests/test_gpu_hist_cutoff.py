"""FP64 histograms that end before the structure does: pairs past nhist are counted per
item and go to the overflow counter.  Counts and overflow equal the oracle's, for one
and several elements, host calls and a plan's structures (each with its own counter)."""
import numpy as np
import pytest

import xansons_hip as xh
import xs_oracle as O
from xansons_hip import structures as st

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [[1], [2], [3000], [900, 1, 1300]])
@pytest.mark.parametrize("part", [0.0, 0.2, 0.6, 0.95])
@pytest.mark.parametrize("bin_", [0.05, 0.0005])
def test_cutoff(counts, part, bin_):
    rng = np.random.default_rng(sum(counts))
    x = rng.uniform(0, 25.0, (3, sum(counts)))
    nh = max(1, int(O.hist_size(x, bin_) * part))
    with xh.Context(0) as ctx:
        print(f"cut-off: {counts} atoms, {nh} bins of {bin_}", flush=True)
        h, ovf = ctx.hist(x, counts, bin_, nh, f64=True)
    ref, ovf_ref = O.hist_f64(x, counts, bin_, nh)
    assert ovf == ovf_ref and np.array_equal(h, ref)


def test_cutoff_in_a_plan():
    ens = st.particle_ensemble(5, seed=3, nmin=100, nmax=3000)
    full = [O.hist_size(e.xyz64(), 0.01) for e in ens]
    nh = [full[0] // 3, full[1], full[2] * 2 // 3, 1, full[4] - 1]
    with xh.Context(0) as ctx:
        print("cut-off: plan", flush=True)
        b = xh.Batch(ctx, [(e.xyz64(), e.el_count) for e in ens], 0.01, nhist=nh)
        hist, _, _ = b.run()
        over = b.overflow()
        for s, e in enumerate(ens):
            ref, ovf = O.hist_f64(e.xyz64(), e.el_count, 0.01, nh[s])
            h0 = int(b.hist_off[s])
            assert np.array_equal(hist[h0:h0 + ref.size], ref.ravel()) and int(over[s]) == ovf, s
        b.close()
