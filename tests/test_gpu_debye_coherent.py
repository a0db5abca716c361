"""Direct Debye sums where every pair has the same distance (the atoms of one element
in one place, those of another in another): the pairs' terms add up without
averaging, so the sum's relative error is a single term's, whatever the number of
pairs, and one bin takes every pair of a run (8,192 x 8,192 atoms: 2^18 a work group).

The bar is a term's, relative to 1/(q r): a few roundings of its phase, as pair by
pair (q R 2^-53 each), the truncation of the series (q R 2^-56 or FP64 rounding), the
moments' resolution of 2^-49 in a few of them, and eps = 1e-8 to first order."""
import numpy as np
import pytest

import xansons_hip as xh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("na,nb", [(1, 1), (64, 65), (1000, 3000), (8192, 8192)])
@pytest.mark.parametrize("q1", [2.0, 20.0])
def test_one_distance(na, nb, q1):
    v = np.array([7.3, -15.1, 4.7])
    x = np.zeros((3, na + nb))
    x[:, na:] = v[:, None]
    q = np.sort(np.random.default_rng(na).uniform(0.3, q1, 300))
    r = np.sqrt((v.astype(np.longdouble) ** 2).sum())
    ph = q.astype(np.longdouble) * r
    ref = np.sin(ph) / (ph + np.longdouble(1e-8))
    with xh.Context(0) as ctx:
        print(f"one distance: {na} x {nb} pairs, q to {q1}", flush=True)
        S = ctx.debye_pairsum(x, [na, nb], q)
    assert not S[0].any() and not S[2].any()
    err = np.abs(S[1].astype(np.longdouble) / (na * nb) - ref) * ph
    qr = float(ph.max())
    bar = max(2.0 ** -52, qr * 2.0 ** -56) + 8 * 2.0 ** -49 + 4 * qr * 2.0 ** -53 + (1e-8 / float(ph.min())) ** 2
    print(f"  {float(err.max()):.2e} of 1/(q r), bar {bar:.2e}", flush=True)
    assert err.max() <= bar
