"""Choice of the class kernels of batched builds: by the batch's quartets together, whatever was built before."""
import pytest

from veloxchem_amd import MolecularBasis, T4CScreener, _native
from veloxchem_amd.workloads import water_cluster

pytestmark = pytest.mark.gpu


def _screener(waters, basis, seed=3):
    mol = water_cluster(waters, 7.0, seed)
    scr = T4CScreener()
    scr.partition(MolecularBasis.read(mol, basis), mol, 'eri')
    return scr


def test_choice_does_not_depend_on_earlier_batches():
    """Batches of one screener on both sides of the line of 2.5e6 quartets, both of more molecules than
    a launch aims at tiled items."""
    scr = _screener(2, 'def2-tzvp')
    quartets = {tuple(c): q for c, q, _, _ in scr.work(12)}
    for cls in ((2, 1, 1, 1), (3, 1, 2, 0), (3, 2, 1, 0)):
        n = 2500000 // quartets[cls]
        assert 512 < n and 2 * n < 65536
        for many in (False, True, False):
            name = _native.batch_class_kernel([scr] * (2 * n if many else n), 12, cls)
            assert ('ksl' in name) == many, (cls, n, name)


def test_one_kernel_per_class_of_uneven_molecules():
    """Molecules on both sides of the line as many of one size would be run a class in one launch."""
    scrs = [_screener(w, 'def2-svp', seed=w) for w in (5, 6, 8, 9)]
    for cls, quartets, _, _ in scrs[-1].work(12):
        if quartets:
            name = _native.batch_class_kernel(scrs, 12, cls)
            assert ' ' not in name, name


def test_small_molecules_of_a_large_batch():
    """One-water molecules beside many larger ones: the class of the launch runs generated, theirs
    matrix-core, since they fill few lanes."""
    big, small = _screener(9, 'def2-svp'), _screener(1, 'def2-svp')
    cls = (2, 1, 1, 1)
    names = _native.batch_class_kernel([big] * 20 + [small] * 20, 12, cls).split()
    assert len(names) == 2 and any('mmd' in k for k in names), names
    assert 'mmd' not in _native.batch_class_kernel([big] * 20, 12, cls)
