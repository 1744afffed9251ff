"""Tiled kernels, both digestions of the matrix-core kernel and the default choice between them,
against the untiled kernels, at the edges of their work items.  The 13 largest classes have no other
kernel than the matrix-core one: its two digestions are checked against the oracle."""
import numpy as np
import pytest

from oracle import oracle as orc
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


@pytest.mark.parametrize('digestion', ['tiles', 'direct'])
@pytest.mark.parametrize('label, omega', [('2jk', 0.0), ('k', 0.4)])
def test_matrix_core_kernel_against_oracle(digestion, label, omega):
    """Every class from la + lb + lc + ld = 4 on, three waters def2-TZVP: 8 + 1 atoms in two groups, so
    that the tiles' items are ragged; direct: as a build of two densities."""
    mol = water_cluster(3, 6.0, 3)
    bas = MolecularBasis.read(mol, 'def2-tzvp')
    scr = T4CScreener()
    scr.partition(bas, mol, 'eri')
    n = bas.get_dimensions_of_basis()
    D = pseudo_density(n, 15, seed=9)
    drv, ctx, lib = FockDriver(), _native.context(), _native.lib()
    name = label + '_rs' if omega else label
    try:
        _native.check(lib.vlx_context_set_variant(ctx, 3))
        if digestion == 'tiles':
            g = np.asarray(drv.compute(scr, D, name, 0.0, omega, 12))
        else:
            ms = Matrices()
            for i in range(2):
                m = make_matrix(bas, mat_t.symmetric)
                m.set_values((i + 1) * D)
                ms.add(m, str(i))
            out = drv.compute(scr, ms, [name] * 2, 0.0, omega, 12)
            g = out.matrix('0').to_numpy()
            assert np.max(np.abs(out.matrix('1').to_numpy() - 2 * g)) <= 2 * n * EPS * np.max(np.abs(2 * g))
    finally:
        _native.check(lib.vlx_context_set_variant(ctx, -1))
    ob = orc.basis_from(bas, mol)
    ref = orc.fock_erf(ob, D, label, 0.0, omega, 12)[0] if omega else orc.fock(ob, D, label, 0.0, 12)[0]
    # n^2 products in orders of their own (n eps on either side), each integral off by some 32 eps
    err = np.max(np.abs(g - ref))
    assert err <= (2 * n + 32) * EPS * max(1.0, np.max(np.abs(ref))), err


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


@pytest.mark.parametrize('mode', ['mixed', 'screened'])
def test_fast_modes_of_large_launches(mode):
    """The same launches in mixed precision (FP32 quartets add 1e-3 tau at most, as in the small
    molecules' test) and with density-weighted screening (1e4 tau)."""
    mol = water_cluster(36, 2.7 * 36 ** (1.0 / 3.0), 3)
    bas = MolecularBasis.read(mol, 'def2-tzvp')
    scr = T4CScreener()
    scr.partition(bas, mol, 'eri')
    D = pseudo_density(bas.get_dimensions_of_basis(), 180, seed=9)
    drv = FockDriver()
    ref = np.asarray(drv.compute(scr, D, '2jk', 0.0, 0.0, 12))
    try:
        if mode == 'mixed':
            _native.set_precision('mixed', 1e-6)
        else:
            _native.set_density_screening(1e-10)
        g = np.asarray(drv.compute(scr, D, '2jk', 0.0, 0.0, 12))
    finally:
        _native.set_precision('fp64')
        _native.set_density_screening(0.0)
    assert np.isfinite(g).all()
    assert np.max(np.abs(g - ref)) <= (1e-9 if mode == 'mixed' else 1e-6)
