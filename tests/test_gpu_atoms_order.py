"""The ensemble builder where its routes part: 16 and 17 (element, block) keys (counted
or sorted), candidates around a work group of 256 and more work groups than one step
of the count's sum (2,048 of two elements), cells just below and above the number of
pairs merged on the host, cut-offs that leave nothing or everything, and an atom set's
memory used again by a smaller and a larger one.

Element counts and order equal the oracle's; positions without displacements bit for
bit, with them within 1e-12 A (ulps of sin, cos and log times a few A)."""
import os
import sys

import numpy as np
import pytest
try:
    import torch  # noqa: F401  (first import can take a minute on a fresh box)
except ImportError:
    torch = None

from conftest import REPO

sys.path.insert(0, os.path.join(REPO, "oracle"))
import xs_oracle as O  # noqa: E402
import xansons_hip as xh  # noqa: E402
from xansons_hip.atoms import Atoms, Block  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = xh.Context(0)
    yield c
    c.close()


def block(seed, n_el, natom, ncell, nsymm=1, sd=0.0, occ=True, **kw):
    rng = np.random.default_rng(seed)
    cell = np.diag([9.0, 8.0, 7.0])
    return Block(r_atom=rng.uniform(0, 1, (natom, 3)) @ cell, el=rng.integers(0, n_el, natom).astype(np.uint32),
                 occ=rng.uniform(0.4, 1.0, natom) if occ else np.ones(natom), dev=np.full(natom, sd),
                 p_symm=np.stack([np.eye(3) * (1 - 2 * (k % 2)) for k in range(nsymm)]),
                 r_symm=rng.uniform(0, 4, (nsymm, 3)), cell=cell, ncell=ncell, **kw)


def check(ctx, blocks, n_el, exact):
    el, blk, xyz = O.calc_atoms(blocks, 21)
    want = xyz[np.argsort(el, kind="stable")]
    print(f"atoms: {len(blocks)} blocks, {n_el} elements, {len(want)} atoms", flush=True)
    a = Atoms(ctx, blocks, n_el, 21)
    try:
        got = a.xyz().T
        assert (a.el_count == np.bincount(el, minlength=n_el)).all()
        per = np.zeros((len(blocks), n_el), np.int64)
        np.add.at(per, (blk, el), 1)
        assert (a.block_el_count == per).all()
    finally:
        a.close()
    assert got.shape == want.shape
    if exact:
        assert (got.copy().view(np.uint64) == want.copy().view(np.uint64)).all()
    elif len(want):
        assert np.abs(got - want).max() <= 1e-12


@pytest.mark.parametrize("n_el,nblocks", [(1, 1), (2, 8), (16, 1), (17, 1), (1, 17), (6, 3)])
def test_keys(ctx, n_el, nblocks):
    check(ctx, [block(b, n_el, 20 + b, (3, 2, 4)) for b in range(nblocks)], n_el, exact=True)


@pytest.mark.parametrize("natom,ncell", [(1, (1, 1, 1)), (1, (1, 1, 255)), (1, (16, 4, 4)), (1, (1, 257, 1)),
                                         (40, (24, 24, 25))])
def test_work_groups(ctx, natom, ncell):
    check(ctx, [block(5, 2, natom, ncell, sd=0.06)], 2, exact=False)


@pytest.mark.parametrize("natom", [32, 33, 60])  # 62,000, 66,000 and 221,250 tests
def test_merge(ctx, natom):
    check(ctx, [block(natom, 3, natom, (2, 3, 2))], 3, exact=True)


@pytest.mark.parametrize("rcut", [1e-3, 12.0, 500.0])
@pytest.mark.parametrize("mol", [False, True])
def test_cutoffs(ctx, rcut, mol):
    kw = dict(mol_rotation=True, dev_mol=0.1) if mol else {}
    check(ctx, [block(9, 2, 12, (4, 4, 4), nsymm=2, sd=0.05, rcut=rcut, **kw)], 2, exact=False)


def test_memory_again(ctx):
    for n in (6, 3, 8, 2):
        check(ctx, [block(n, 2, 10, (n, n, n))], 2, exact=True)
