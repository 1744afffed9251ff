"""vlx_fock_compute_device_noalloc: the build whose F' accumulator lives in the library's static
device scratch, against vlx_fock_compute_device (the allocating entry point) on the same
device-resident inputs, through the C ABI.  Two calls in a row, the second on a smaller
molecule (the scratch keeps the first call's contents, so the second also checks the clear),
plus the argument checks: a screener without a prepared schedule and a basis above the
scratch limit are refused with VLX_ERR_ARG."""
import ctypes

import numpy as np
import pytest

from veloxchem_amd import MolecularBasis, T4CScreener, _native
from veloxchem_amd.workloads import pseudo_density, water_cluster

pytestmark = pytest.mark.gpu


def _case(nmol, box, seed, basis='def2-svp'):
    mol = water_cluster(nmol, box, seed)
    bas = MolecularBasis.read(mol, basis)
    scr = T4CScreener()
    scr.partition(bas, mol, 'eri')
    n = bas.get_dimensions_of_basis()
    return scr, pseudo_density(n, 5 * nmol, seed=seed + 1), n


def _builds(scr, D, n, label=b'2jk', xf=1.0, ithr=12):
    lib, ctx = _native.lib(), _native.context(0)
    d_dm, d_a, d_b = _native.DeviceArray((n, n)), _native.DeviceArray((n, n)), _native.DeviceArray((n, n))
    try:
        d_dm.upload(D)
        # the allocating build prepares the screener's schedule, then the scratch build reuses it
        _native.check(lib.vlx_fock_compute_device(ctx, scr.handle, d_dm.ptr, label, xf, 0.0, ithr, d_a.ptr))
        _native.check(lib.vlx_fock_compute_device_noalloc(ctx, scr.handle, d_dm.ptr, label, xf, 0.0, ithr, d_b.ptr))
        _native.check(lib.vlx_context_synchronize(ctx))
        return d_a.download(), d_b.download()
    finally:
        for a in (d_dm, d_a, d_b):
            a.free()


def test_noalloc_matches_allocating_build_twice():
    big = _case(6, 7.0, 41)
    small = _case(2, 4.0, 43)
    for (scr, D, n), label, xf in ((big, b'2jk', 1.0), (small, b'2jkx', 0.37)):
        print(f'noalloc: {n} AOs, label {label.decode()}', flush=True)
        ga, gb = _builds(scr, D, n, label, xf)
        err = float(np.max(np.abs(ga - gb)))
        print(f'  max|G_noalloc - G| = {err:.3e}', flush=True)
        assert np.all(np.isfinite(gb))
        assert err < 1e-10
        assert np.max(np.abs(gb - gb.T)) < 1e-12


def test_noalloc_mixed_precision_matches():
    scr, D, n = _case(3, 5.0, 47)
    _native.set_precision('mixed', 1e-7)
    try:
        ga, gb = _builds(scr, D, n)
    finally:
        _native.set_precision('fp64')
    assert float(np.max(np.abs(ga - gb))) < 1e-10


def test_noalloc_after_a_build_of_several_densities():
    """The schedule of a build of several densities serves the no-allocation build too."""
    lib, ctx = _native.lib(), _native.context(0)
    scr, D, n = _case(2, 4.0, 57, 'def2-tzvp')
    d_dm, d_two, d_g = _native.DeviceArray((2, n, n)), _native.DeviceArray((2, n, n)), _native.DeviceArray((n, n))
    try:
        d_dm.upload(np.stack([D, 2.0 * D]))
        labels = (ctypes.c_char_p * 2)(b'2jk', b'k')
        _native.check(lib.vlx_fock_compute_multi_device(ctx, scr.handle, 2, d_dm.ptr, None, labels, 0.0, 0.0, 12,
                                                        d_two.ptr))
        _native.check(lib.vlx_fock_compute_device_noalloc(ctx, scr.handle, d_dm.ptr, b'2jk', 0.0, 0.0, 12, d_g.ptr))
        _native.check(lib.vlx_context_synchronize(ctx))
        two, g = d_two.download(), d_g.download()
    finally:
        for a in (d_dm, d_two, d_g):
            a.free()
    # sums of up to n^2 products in orders of their own: n eps on either side
    assert np.max(np.abs(g - two[0])) <= 2 * n * np.finfo(float).eps * np.max(np.abs(two[0]))


def test_noalloc_refuses_unprepared_schedule_and_large_basis():
    lib, ctx = _native.lib(), _native.context(0)
    scr, D, n = _case(1, 3.0, 51)
    d_dm, d_g = _native.DeviceArray((n, n)), _native.DeviceArray((n, n))
    try:
        d_dm.upload(D)
        # ithreshold 11 was never built for this screener: no schedule, no build
        with pytest.raises(ValueError, match='schedule'):
            _native.check(lib.vlx_fock_compute_device_noalloc(ctx, scr.handle, d_dm.ptr, b'2jk', 1.0, 0.0, 11,
                                                              d_g.ptr))
    finally:
        d_dm.free()
        d_g.free()
    # 128 waters in def2-SVP: 3072 AOs is the limit, 3096 is above it (the check comes before any launch)
    big, _, nbig = _case(129, 20.0, 53)
    assert nbig > 3072
    dummy = ctypes.c_void_p(1)
    with pytest.raises(ValueError, match='scratch limit'):
        _native.check(lib.vlx_fock_compute_device_noalloc(ctx, big.handle, dummy, b'2jk', 1.0, 0.0, 12, dummy))
