"""Builds captured into a HIP graph on the context's stream, after an eager build of another kind."""
import ctypes

import numpy as np
import pytest

from veloxchem_amd import FockDriver, MolecularBasis, T4CScreener, _native
from veloxchem_amd.workloads import pseudo_density, water_cluster

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('first, label', [('2jk', 'j'), ('two densities', '2jk')])
def test_capture_after_another_build(first, label):
    """A Coulomb build whose lists do not exist yet, and a build whose screener has only the schedule of
    several densities: nothing is allocated under capture, and every replay gives the eager result."""
    import torch
    mol = water_cluster(2, 4.0, 5)
    bas = MolecularBasis.read(mol, 'def2-tzvp')
    scr, ref_scr = T4CScreener(), T4CScreener()
    scr.partition(bas, mol, 'eri')
    ref_scr.partition(bas, mol, 'eri')
    n = bas.get_dimensions_of_basis()
    dens = [pseudo_density(n, 10, seed=s) for s in (1, 2, 3)]
    lib, ctx = _native.lib(), _native.context()
    d = torch.from_numpy(np.stack(dens[:2])).to('cuda:0')
    g = torch.zeros_like(d)
    torch.cuda.synchronize()

    def ptr(t):
        return ctypes.c_void_p(t.data_ptr())

    def build(lab):
        _native.check(lib.vlx_fock_compute_device(ctx, scr.handle, ptr(d[0]), lab.encode(), 0.0, 0.0, 12, ptr(g[0])))
    if first == 'two densities':
        labels = (ctypes.c_char_p * 2)(b'2jk', b'k')
        _native.check(lib.vlx_fock_compute_multi_device(ctx, scr.handle, 2, ptr(d), None, labels, 0.0, 0.0, 12, ptr(g)))
        # the F' accumulator of single builds
        _native.check(lib.vlx_fock_compute_device(ctx, ref_scr.handle, ptr(d[0]), b'2jk', 0.0, 0.0, 12, ptr(g[0])))
    else:
        build(first)
    _native.check(lib.vlx_context_synchronize(ctx))
    stream = torch.cuda.ExternalStream(lib.vlx_context_stream(ctx))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode='thread_local'):
        build(label)
    for D in dens:
        d[0].copy_(torch.from_numpy(D))
        g.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        got = g[0].cpu().numpy()
        # an eager build between the replays
        ref = np.asarray(FockDriver().compute(ref_scr, D, label, 0.0, 0.0, 12))
        # sums of up to n^2 products in orders of their own: n eps on either side
        assert np.max(np.abs(got - ref)) <= 2 * n * np.finfo(float).eps * max(1.0, np.max(np.abs(ref)))
