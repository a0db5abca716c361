"""FP64 histograms whose tile pairs have about as many pairs as are taken one by one
(512): tiles of 16 and 17 atoms (an I unit is two tiles), of one atom, own tiles and
tiles of two elements, unequal ones, with and without pairs past the last bin, and
enough atoms for the items to be shared out.  Counts and overflow equal the oracle's."""
import numpy as np
import pytest

import xansons_hip as xh
import xs_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts,edge,bin_", [
    ([1], 1.0, 0.1), ([2], 1.0, 0.1), ([15], 5.0, 0.1), ([16], 5.0, 0.1), ([31], 5.0, 0.1),
    ([32], 5.0, 0.1), ([33], 5.0, 0.1), ([22, 23, 24], 5.0, 0.01), ([1, 511, 512, 513], 12.0, 0.01),
    ([256, 3], 9.0, 0.01), ([171, 3], 9.0, 0.01), ([4000], 20.0, 2e-4),      # tiles of a few atoms
    ([1000, 1500], 1500.0, 1e-3),  # tiles of one
])
@pytest.mark.parametrize("part", [1.0, 0.5])
def test_few(counts, edge, bin_, part):
    rng = np.random.default_rng(sum(counts))
    x = rng.uniform(0, edge, (3, sum(counts)))
    nh = max(1, int(O.hist_size(x, bin_) * part))
    with xh.Context(0) as ctx:
        print(f"few: {counts} atoms, {nh} bins of {bin_}", flush=True)
        h, ovf = ctx.hist(x, counts, bin_, nh, f64=True)
        b = xh.Batch(ctx, [(x, counts)], bin_, nhist=[nh])
        hb, _, _ = b.run()
        over = int(b.overflow()[0])
        b.close()
    ref, ovf_ref = O.hist_f64(x, counts, bin_, nh)
    assert ovf == ovf_ref and np.array_equal(h, ref)
    assert over == ovf_ref and np.array_equal(hb, ref.ravel())


def test_cluster_with_a_halo():
    """Full tiles next to tiles of one atom, in one item's run."""
    rng = np.random.default_rng(4)
    v = rng.normal(size=(3, 4000))
    v /= np.linalg.norm(v, axis=0)
    x = v * (3 * rng.pareto(1.5, 4000).clip(0, 60))
    nh = O.hist_size(x, 2e-3)
    with xh.Context(0) as ctx:
        print(f"halo: {nh} bins", flush=True)
        h, ovf = ctx.hist(x, [2500, 1500], 2e-3, nh, f64=True)
    ref, _ = O.hist_f64(x, [2500, 1500], 2e-3, nh)
    assert ovf == 0 and np.array_equal(h, ref)
