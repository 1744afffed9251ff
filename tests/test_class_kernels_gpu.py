"""Tiled kernels, both digestions of the matrix-core kernel and the default choice between them,
against the untiled kernels, at the edges of their work items."""
import numpy as np
import pytest

from veloxchem_amd import FockDriver, Matrices, MolecularBasis, T4CScreener, _native, make_matrix, mat_t
from veloxchem_amd.workloads import pseudo_density, water_cluster

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


@pytest.mark.parametrize('waters, basis, label, omega, ithreshold', [
    (1, 'def2-svp', '2jk', 0.0, 12),      # one atom group, chunks of a few kets, one molecule's latency
    (1, 'def2-tzvp', '2jkx', 0.0, -1),    # no screening, f shells, every rank of the same-class pairs
    (3, 'def2-svpd', 'k', 0.0, 12),       # several groups of 6 atoms, the last one of 3
    (5, 'def2-svp', 'j', 0.0, 10),        # 12 + 3 atoms, J tiles only
    (5, 'def2-svp', 'kx_rs', 0.4, 12),    # attenuated exchange
    (6, 'def2-tzvp', '2jk', 0.0, 12),     # (pp|pp) chunks past 64 entries, items of several chunks
    # Coulomb builds: the default choice goes through Hermite densities
    (1, 'def2-svp', 'j', 0.0, 12),        # ranks of fewer entries than a block, one stage of kets
    (2, 'def2-tzvp', 'j_rs', 0.5, 12),    # f shells: ranks 0 to 6, attenuated
    (3, 'def2-svpd', 'j', 0.0, 6),        # bras that meet no ket of some ranks
    (4, 'def2-tzvp', 'j', 0.0, 12),       # ragged last blocks and stages
    (2, 'def2-svp', 'j', 0.0, -1),        # unscreened: the class kernels
])
def test_class_kernels_agree(waters, basis, label, omega, ithreshold):
    mol = water_cluster(waters, 6.0, 3)
    bas = MolecularBasis.read(mol, basis)
    scr = T4CScreener()
    scr.partition(bas, mol, 'eri')
    n = bas.get_dimensions_of_basis()
    D = pseudo_density(n, 5 * waters, seed=9)
    mats = {}
    drv, ctx, lib = FockDriver(), _native.context(), _native.lib()
    # an element sums up to n^2 products I D in an order of each kernel's own; the rounding errors of
    # n^2 terms are independent, so they grow as n eps on each side
    try:
        for v in (0, -1, 1, 2, 3, 4, 5, 6):
            _native.check(lib.vlx_context_set_variant(ctx, v))
            mats[v] = np.asarray(drv.compute(scr, D, label, 0.5, omega, ithreshold))
    finally:
        _native.check(lib.vlx_context_set_variant(ctx, -1))
    tol = 2 * n * EPS * max(1.0, np.max(np.abs(mats[0])))
    for v, g in mats.items():
        assert np.isfinite(g).all(), v
        assert np.max(np.abs(g - mats[0])) <= tol, (v, np.max(np.abs(g - mats[0])), tol)


def test_direct_digestion_of_matrix_core_classes():
    """Two densities in one call digest directly; each is the single build (LDS tiles)."""
    mol = water_cluster(2, 6.0, 3)
    bas = MolecularBasis.read(mol, 'def2-tzvp')
    scr = T4CScreener()
    scr.partition(bas, mol, 'eri')
    n = bas.get_dimensions_of_basis()
    dens = [pseudo_density(n, 10, seed=s) for s in (1, 2)]
    drv, ctx, lib = FockDriver(), _native.context(), _native.lib()
    try:
        _native.check(lib.vlx_context_set_variant(ctx, 3))
        ms = Matrices()
        for i, d in enumerate(dens):
            m = make_matrix(bas, mat_t.symmetric)
            m.set_values(d)
            ms.add(m, str(i))
        out = drv.compute(scr, ms, ['2jk', 'k'], 0.0, 0.0, 12)
        for i, lab in enumerate(['2jk', 'k']):
            one = np.asarray(drv.compute(scr, dens[i], lab, 0.0, 0.0, 12))
            g = out.matrix(str(i)).to_numpy()
            assert np.max(np.abs(g - one)) <= 2 * n * EPS * max(1.0, np.max(np.abs(one)))
    finally:
        _native.check(lib.vlx_context_set_variant(ctx, -1))


def test_default_kernels_of_large_launches():
    """2.5e6 quartets and more in several classes: the default there against the untiled kernels."""
    mol = water_cluster(36, 2.7 * 36 ** (1.0 / 3.0), 3)
    bas = MolecularBasis.read(mol, 'def2-tzvp')
    scr = T4CScreener()
    scr.partition(bas, mol, 'eri')
    n = bas.get_dimensions_of_basis()
    D = pseudo_density(n, 180, seed=9)
    drv, ctx, lib = FockDriver(), _native.context(), _native.lib()
    g = np.asarray(drv.compute(scr, D, '2jk', 0.0, 0.0, 12))
    names = {c: _native.class_kernel(scr, 12, c) for c in ((2, 1, 1, 1), (3, 0, 3, 0), (3, 0, 2, 0))}
    try:
        _native.check(lib.vlx_context_set_variant(ctx, 0))
        ref = np.asarray(drv.compute(scr, D, '2jk', 0.0, 0.0, 12))
    finally:
        _native.check(lib.vlx_context_set_variant(ctx, -1))
    assert any('ksl' in k for k in names.values()), names
    assert np.max(np.abs(g - ref)) <= 2 * n * EPS * max(1.0, np.max(np.abs(ref)))
