"""Timed cases of the two-electron Fock build and of the learned guess's network.

The cases are what a program built on this package asks of it: one Fock build per call, on host
arrays through ``FockDriver.compute`` (the drop-in call) or on matrices that stay on the device
through ``vlx_fock_compute_device`` (what the SCF loop does every iteration), several densities or
several molecules in one call, and the training step of the starting-density network.  Molecules are
seeded water clusters at the density of the repository's 32- and 64-water workloads; every build uses
the kernels the library picks by itself (no autotuner pass).

``exact`` is an independent evaluation in float64: McMurchie-Davidson integrals over the shell table,
all of them (no Schwarz selection), contracted with the density.
"""
import ctypes
import functools
import math

import numpy as np
import torch

from veloxchem_amd import (FockDriver, Matrices, MolecularBasis, T4CScreener, _native, make_matrix, mat_t)
from veloxchem_amd.densitynet import DensityNet
from veloxchem_amd.sadguess import sad_density
from veloxchem_amd.workloads import water_cluster

# eri_thresh 1e-12, the SCF driver's default
ITHRESHOLD = 12
# labels with their digestion: (Coulomb factor, exchange factor or None for the caller's, erf operator)
LABELS = {'2jk': (2.0, -1.0, False), '2jkx': (2.0, None, False), 'j': (1.0, 0.0, False), 'k': (0.0, 1.0, False),
          'kx_rs': (0.0, None, True), 'j_rs': (1.0, 0.0, True)}
# the learned guess's network: 70 inputs, two hidden layers of 256, 14 x 14 blocks (def2-SVP)
N_IN, N_HIDDEN, BLOCK = 70, 256, 14


def listed():
    return [
        # smallest call: one molecule on host arrays, as the first thing a user tries; launch latency
        {'name': 'water_svp_host', 'kind': 'host', 'waters': 1, 'basis': 'def2-svp', 'label': '2jk', 'xf': 1.0,
         'omega': 0.0},
        # long-range exchange of a range-separated hybrid functional, with f shells
        {'name': 'w2_tzvp_kxrs_host', 'kind': 'host', 'waters': 2, 'basis': 'def2-tzvp', 'label': 'kx_rs', 'xf': 0.21,
         'omega': 0.33},
        # an SCF iteration of a small cluster, matrices on the device
        {'name': 'w8_svp_2jk', 'kind': 'device', 'waters': 8, 'basis': 'def2-svp', 'label': '2jk', 'xf': 1.0,
         'omega': 0.0},
        # hybrid functional with diffuse functions, an odd cluster size
        {'name': 'w13_svpd_2jkx', 'kind': 'device', 'waters': 13, 'basis': 'def2-svpd', 'label': '2jkx', 'xf': 0.2,
         'omega': 0.0},
        # the 32-water workload of the benchmark (768 AOs)
        {'name': 'w32_svp_2jk', 'kind': 'device', 'waters': 32, 'basis': 'def2-svp', 'label': '2jk', 'xf': 1.0,
         'omega': 0.0},
        # a triple-zeta SCF iteration of middle size (860 AOs)
        {'name': 'w20_tzvp_2jk', 'kind': 'device', 'waters': 20, 'basis': 'def2-tzvp', 'label': '2jk', 'xf': 1.0,
         'omega': 0.0},
        # Coulomb matrix only: pure density functionals
        {'name': 'w27_tzvp_j', 'kind': 'device', 'waters': 27, 'basis': 'def2-tzvp', 'label': 'j', 'xf': 0.0,
         'omega': 0.0},
        # largest: the benchmark's 64-water def2-TZVP size (2752 AOs)
        {'name': 'w64_tzvp_2jk', 'kind': 'device', 'waters': 64, 'basis': 'def2-tzvp', 'label': '2jk', 'xf': 1.0,
         'omega': 0.0},
        # mixed precision: recursions in FP32 below the Schwarz x max|D| bound
        {'name': 'w16_svp_mixed', 'kind': 'mixed', 'waters': 16, 'basis': 'def2-svp', 'label': '2jk', 'xf': 1.0,
         'omega': 0.0, 'tau': 1e-6},
        # response solver: several trial densities, symmetric and general, in one pass over the integrals
        {'name': 'w6_svp_multi4', 'kind': 'multi', 'waters': 6, 'basis': 'def2-svp', 'densities': 4},
        # many small molecules in one call
        {'name': 'batch40_svp', 'kind': 'batch', 'molecules': 40, 'most': 9, 'basis': 'def2-svp', 'label': '2jk'},
        # one training step of the starting-density network
        {'name': 'guess_train', 'kind': 'train', 'batch': 2048},
    ]


def draw(rng):
    kind = rng.choice(['host', 'device', 'device', 'device', 'mixed', 'multi', 'batch', 'train'])

    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if kind == 'train':
        return {'kind': kind, 'batch': size(33, 4096)}
    if kind == 'batch':
        return {'kind': kind, 'molecules': size(3, 60), 'most': rng.randint(2, 9), 'basis': 'def2-svp',
                'label': rng.choice(['2jk', 'j', 'k'])}
    if kind == 'multi':
        return {'kind': kind, 'waters': size(1, 12), 'basis': rng.choice(['def2-svp', 'def2-svpd']),
                'densities': rng.randint(2, 6)}
    basis = rng.choice(['def2-svp', 'def2-svpd', 'def2-tzvp'])
    most = {'def2-svp': 48, 'def2-svpd': 24, 'def2-tzvp': 40}[basis]
    if kind == 'mixed':
        return {'kind': kind, 'waters': size(2, most), 'basis': basis, 'label': '2jk', 'xf': 1.0, 'omega': 0.0,
                'tau': rng.choice([1e-6, 1e-8])}
    label = rng.choice(['2jk', '2jk', '2jkx', 'j', 'k', 'kx_rs', 'j_rs'])
    return {'kind': kind, 'waters': size(1, 10 if kind == 'host' else most), 'basis': basis, 'label': label,
            'xf': round(rng.uniform(0.1, 0.8), 2), 'omega': round(rng.uniform(0.2, 0.5), 2)}


# ---- inputs ------------------------------------------------------------------------------------


def _cluster(waters, seed):
    return water_cluster(waters, max(2.7, 10.0 * (waters / 32.0) ** (1.0 / 3.0)), seed)


def _density(mol, bas, rng, general=False, trial=False):
    """A density as the SCF loop has it on its way: the superposition of atomic densities plus
    overlap-like off-diagonal elements that fall off with the distance of the atoms; ``trial``: the
    second part alone, as response solvers have."""
    n = bas.get_dimensions_of_basis()
    sh = bas.shell_arrays(mol.get_coordinates_in_bohr())
    xyz = np.zeros((n, 3))
    for s in range(len(sh['l'])):
        for m in range(2 * sh['l'][s] + 1):
            xyz[sh['ao_base'][s] + m * sh['ao_stride'][s]] = np.asarray(sh['centers']).reshape(-1, 3)[s]
    dist = np.sqrt(np.maximum(0.0, ((xyz[:, None, :] - xyz[None, :, :]) ** 2).sum(-1)))
    x = rng.normal(size=(n, n)) * 0.05 * np.exp(-0.7 * dist)
    if not general:
        x = 0.5 * (x + x.T)
    if trial:
        return np.ascontiguousarray(x)
    return np.ascontiguousarray(sad_density(mol, MolecularBasis.read(mol, 'ao-start-guess'), bas) + x)


def _molecule(case, seed):
    mol = _cluster(case['waters'], seed)
    bas = MolecularBasis.read(mol, case['basis'])
    return mol, bas


def _screener(mol, bas):
    scr = T4CScreener()
    scr.partition(bas, mol, 'eri')
    return scr


MULTI_LABELS = ('2jk', 'j', 'k', '2jkx')
MULTI_XF = 0.2


def _multi_densities(case, mol, bas, rng):
    """Labels, flags (general or symmetric) and arrays of the trial densities."""
    got = []
    for i in range(case['densities']):
        general = i % 2 == 1
        got.append((MULTI_LABELS[(i // 2) % 4], general, _density(mol, bas, rng, general=general, trial=True)))
    return got


def _batch_sizes(case):
    """Waters of each molecule: 1 .. most, the same for every seed."""
    rng = np.random.Generator(np.random.PCG64(100 * case['molecules'] + case['most']))
    return [int(w) for w in rng.integers(1, case['most'] + 1, case['molecules'])]


def _batch_molecules(case, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    got = []
    for k, waters in enumerate(_batch_sizes(case)):
        mol = _cluster(waters, seed + 1 + k)
        bas = MolecularBasis.read(mol, case['basis'])
        got.append((mol, bas, _density(mol, bas, rng)))
    return got


def _train_inputs(case, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    m = case['batch']
    x = rng.normal(size=(m, N_IN)).astype(np.float32) * 0.5
    x[:, :26] = rng.random((m, 26)) < 0.08  # one-hot pair features
    t = rng.normal(size=(m, BLOCK * BLOCK)).astype(np.float32) * 0.03
    shape = rng.choice([5, 14], size=(m, 2)).astype(np.int32)
    params = []
    for fi, fo in ((N_IN, N_HIDDEN), (N_HIDDEN, N_HIDDEN), (N_HIDDEN, BLOCK * BLOCK)):
        params += [rng.normal(size=fi * fo) * math.sqrt(2.0 / fi) * 0.5, rng.normal(size=fo) * 0.02]
    return x, t, shape, np.concatenate(params).astype(np.float32)


def prepare(case, seed):
    kind = case['kind']
    if kind == 'train':
        x, t, shape, params = _train_inputs(case, seed)
        net = DensityNet(N_IN, N_HIDDEN, BLOCK * BLOCK, BLOCK, case['batch'])
        net.set_params(params)
        dev = 'cuda:0'
        return {'kind': kind, 'net': net, 'x': torch.from_numpy(x).to(dev), 't': torch.from_numpy(t).to(dev),
                'shape': torch.from_numpy(shape).to(dev)}
    if kind == 'batch':
        mols = _batch_molecules(case, seed)
        scrs = [_screener(m, b) for m, b, _ in mols]
        dens = [torch.from_numpy(d).to('cuda:0') for _, _, d in mols]
        outs = [torch.empty_like(d) for d in dens]
        torch.cuda.synchronize()
        arr = ctypes.c_void_p * len(mols)
        return {'kind': kind, 'screeners': scrs, 'dens': dens, 'outs': outs, 'label': case['label'].encode(),
                'handles': arr(*[s.handle.value for s in scrs]), 'd_ptrs': arr(*[d.data_ptr() for d in dens]),
                'g_ptrs': arr(*[g.data_ptr() for g in outs]), 'lib': _native.lib(), 'ctx': _native.context(0)}
    mol, bas = _molecule(case, seed)
    rng = np.random.Generator(np.random.PCG64(seed + 7))
    state = {'kind': kind, 'screener': _screener(mol, bas), 'case': case}
    if kind == 'multi':
        mats, labels = Matrices(), []
        for i, (label, general, d) in enumerate(_multi_densities(case, mol, bas, rng)):
            mat = make_matrix(bas, mat_t.general if general else mat_t.symmetric)
            mat.set_values(d)
            mats.add(mat, str(i))
            labels.append(label)
        state.update(driver=FockDriver(), mats=mats, labels=labels)
        return state
    d = _density(mol, bas, rng)
    if kind == 'host':
        mat = make_matrix(bas, mat_t.symmetric)
        mat.set_values(d)
        state.update(driver=FockDriver(), density=mat)
        return state
    state['density'] = torch.from_numpy(d).to('cuda:0')
    state['out'] = torch.empty_like(state['density'])
    torch.cuda.synchronize()
    state.update(lib=_native.lib(), ctx=_native.context(0), label=case['label'].encode())
    return state


# ---- one pass ----------------------------------------------------------------------------------


def run(state):
    kind = state['kind']
    if kind == 'train':
        net = state['net']
        loss, grad = net.loss_grad(state['x'], state['t'], state['shape'], want_grad=True)
        return {'loss': loss, 'grad': grad}
    if kind == 'batch':
        _native.check(state['lib'].vlx_fock_compute_batch_device(
            state['ctx'], len(state['outs']), state['handles'], state['d_ptrs'], state['label'], 1.0, 0.0, ITHRESHOLD,
            state['g_ptrs']))
        return state['outs']
    case = state['case']
    if kind == 'multi':
        out = state['driver'].compute(state['screener'], state['mats'], state['labels'], MULTI_XF, 0.0, ITHRESHOLD)
        return [out.matrix(k).to_numpy() for k in out.keys()]
    if kind == 'host':
        return state['driver'].compute(state['screener'], state['density'], case['label'], case['xf'], case['omega'],
                                       ITHRESHOLD).to_numpy()
    if kind == 'mixed':
        _native.set_precision('mixed', case['tau'])
    _native.check(state['lib'].vlx_fock_compute_device(
        state['ctx'], state['screener'].handle, ctypes.c_void_p(state['density'].data_ptr()), state['label'],
        case['xf'], case['omega'], ITHRESHOLD, ctypes.c_void_p(state['out'].data_ptr())))
    if kind == 'mixed':
        _native.set_precision('fp64')
    return state['out']


# ---- what a pass cannot do without -------------------------------------------------------------


@functools.lru_cache(maxsize=None)
def _cluster_work(waters, basis, seed=1):
    """(AOs, primitive pairs, per class (L, integrals, quartets, primitive quartets)) of one build."""
    mol, bas = _molecule({'waters': waters, 'basis': basis}, seed)
    sh = bas.shell_arrays(mol.get_coordinates_in_bohr())
    prims = int(sum(sh['nprim']))
    classes = [(sum(c), math.prod(2 * x + 1 for x in c), q, pq)
               for c, q, pq, _ in _screener(mol, bas).work(ITHRESHOLD)]
    return bas.get_dimensions_of_basis(), prims * (prims + 1) // 2, classes


def _nherm(ltot):
    return (ltot + 1) * (ltot + 2) * (ltot + 3) // 6


def _build_flops(classes, coulomb, exchange):
    """Set-up, Boys function and Hermite integrals per primitive quartet; digestion per integral."""
    return float(sum(pq * (53 + 4 * ltot + 2 * _nherm(ltot)) + q * nint * (4 * coulomb + 8 * exchange)
                     for ltot, nint, q, pq in classes))


def work(case):
    kind = case['kind']
    if kind == 'train':
        m = case['batch']
        weights = N_IN * N_HIDDEN + N_HIDDEN * N_HIDDEN + N_HIDDEN * BLOCK * BLOCK
        return {'bytes': 4.0 * (m * (N_IN + BLOCK * BLOCK + 2) + 2 * (weights + 2 * N_HIDDEN + BLOCK * BLOCK)),
                'flops': 2.0 * m * (3 * weights - N_IN * N_HIDDEN)}
    if kind == 'batch':
        total = {'bytes': 0.0, 'flops': 0.0}
        _, fk, _ = LABELS[case['label']]
        for waters in _batch_sizes(case):
            n, pp, classes = _cluster_work(waters, case['basis'])
            total['bytes'] += 16.0 * n * n + 64.0 * pp
            total['flops'] += _build_flops(classes, case['label'] != 'k', fk != 0.0)
        return total
    n, pp, classes = _cluster_work(case['waters'], case['basis'])
    if kind == 'multi':
        k = case['densities']
        flops = _build_flops(classes, 0, 0)
        for i in range(k):
            fj, fk, _ = LABELS[MULTI_LABELS[(i // 2) % 4]]
            flops += _build_flops(classes, fj != 0.0, fk != 0.0) - _build_flops(classes, 0, 0)
        return {'bytes': 16.0 * n * n * k + 64.0 * pp, 'flops': flops}
    fj, fk, _ = LABELS[case['label']]
    return {'bytes': 16.0 * n * n + 64.0 * pp, 'flops': _build_flops(classes, fj != 0.0, fk != 0.0)}


def tolerance(case):
    kind = case['kind']
    if kind == 'train':
        # bf16 operands, fp32 sums: 2e-3 off the float64 gradient, four times that
        return {'rel': 8e-3}
    if kind == 'mixed':
        # FP32 recursions for the quartets below tau x max|D|
        return {'rel': 1e-10 if case['tau'] > 1e-7 else 2e-11}
    # FP64 with the Schwarz selection at 1e-12: up to 3.4e-12 off the sum over all quartets
    return {'rel': 1.2e-11}


# ---- float64 evaluation ------------------------------------------------------------------------

# real solid harmonics of one shell as Cartesian terms ((i, j, k), factor), in the AO component order
_S3, _S10, _S15, _S6 = math.sqrt(3.0), math.sqrt(2.5), math.sqrt(15.0), math.sqrt(1.5)
_HARMONICS = {
    0: [[((0, 0, 0), 1.0)]],
    1: [[((0, 1, 0), 1.0)], [((0, 0, 1), 1.0)], [((1, 0, 0), 1.0)]],
    2: [[((1, 1, 0), 2 * _S3)], [((0, 1, 1), 2 * _S3)],
        [((0, 0, 2), 2.0), ((2, 0, 0), -1.0), ((0, 2, 0), -1.0)], [((1, 0, 1), 2 * _S3)],
        [((2, 0, 0), _S3), ((0, 2, 0), -_S3)]],
    3: [[((2, 1, 0), 3 * _S10), ((0, 3, 0), -_S10)], [((1, 1, 1), 2 * _S15)],
        [((0, 1, 2), 4 * _S6), ((2, 1, 0), -_S6), ((0, 3, 0), -_S6)],
        [((0, 0, 3), 2.0), ((2, 0, 1), -3.0), ((0, 2, 1), -3.0)],
        [((1, 0, 2), 4 * _S6), ((3, 0, 0), -_S6), ((1, 2, 0), -_S6)],
        [((2, 0, 1), _S15), ((0, 2, 1), -_S15)], [((3, 0, 0), _S10), ((1, 2, 0), -3 * _S10)]],
}
_EXACT_MOST = 200  # AOs: the whole tensor of integrals is formed
_CHUNK = 1 << 27   # doubles of one block of Hermite integrals


def _hermite_list(ltot):
    return [(t, u, n - t - u) for n in range(ltot + 1) for t in range(n, -1, -1) for u in range(n - t, -1, -1)]


def _boys(top, arg):
    """F_0 .. F_top: the ascending series for F_top and the downward recursion below T = 36, the
    upward recursion from erf above."""
    t = arg.clamp(max=36.0)
    ex = torch.exp(-t)
    term = torch.full_like(t, 1.0 / (2 * top + 1))
    total = term.clone()
    for i in range(1, 160):
        term = term * (2.0 * t) / (2 * top + 2 * i + 1)
        total += term
    small = [None] * (top + 1)
    small[top] = total * ex
    for m in range(top - 1, -1, -1):
        small[m] = (2.0 * t * small[m + 1] + ex) / (2 * m + 1)
    big_t = arg.clamp(min=36.0)
    ex = torch.exp(-big_t)
    f = 0.5 * torch.sqrt(math.pi / big_t) * torch.erf(torch.sqrt(big_t))
    got, low = [], arg < 36.0
    for m in range(top + 1):
        got.append(torch.where(low, small[m], f))
        f = ((2 * m + 1) * f - ex) / (2.0 * big_t)
    return got


def _pair_class(sh, la, lb, device):
    """Shell pairs (A, B), l_A = la, l_B = lb, of the table: AO indices, primitive pairs and their
    Hermite-to-spherical matrices."""
    ls = np.asarray(sh['l'])
    cen = np.asarray(sh['centers']).reshape(-1, 3)
    pairs = [(a, b) for a in np.where(ls == la)[0] for b in np.where(ls == lb)[0] if la != lb or a >= b]
    if not pairs:
        return None
    owner, ea, eb, ca, cb, ra, rb = [], [], [], [], [], [], []
    for k, (a, b) in enumerate(pairs):
        oa, ob = sh['prim_offset'][a], sh['prim_offset'][b]
        for i in range(sh['nprim'][a]):
            for j in range(sh['nprim'][b]):
                owner.append(k)
                ea.append(sh['exps'][oa + i])
                eb.append(sh['exps'][ob + j])
                ca.append(sh['norms'][oa + i])
                cb.append(sh['norms'][ob + j])
                ra.append(cen[a])
                rb.append(cen[b])

    def dev(v):
        return torch.tensor(np.array(v), dtype=torch.float64, device=device)

    a, b, ra, rb = dev(ea), dev(eb), dev(ra), dev(rb)
    p = a + b
    centre = (a[:, None] * ra + b[:, None] * rb) / p[:, None]
    ab2 = ((ra - rb) ** 2).sum(1)
    pref = dev(ca) * dev(cb) * torch.exp(-a * b / p * ab2)
    # one-dimensional Hermite coefficients e[axis][i][j][t]
    e = []
    for x in range(3):
        pa, pb, h = centre[:, x] - ra[:, x], centre[:, x] - rb[:, x], 0.5 / p
        g = {(0, 0): [torch.ones_like(p)]}
        for i in range(la + 1):
            for j in range(lb + 1):
                if (i, j) == (0, 0):
                    continue
                src, shift = (g[(i - 1, j)], pa) if j == 0 else (g[(i, j - 1)], pb)
                new = []
                for t in range(i + j + 1):
                    v = torch.zeros_like(p)
                    if t < len(src):
                        v = v + shift * src[t]
                    if t > 0:
                        v = v + h * src[t - 1]
                    if t + 1 < len(src):
                        v = v + (t + 1) * src[t + 1]
                    new.append(v)
                g[(i, j)] = new
        e.append(g)
    herm = {h: k for k, h in enumerate(_hermite_list(la + lb))}
    u = torch.zeros(len(owner), len(herm), (2 * la + 1) * (2 * lb + 1), dtype=torch.float64, device=device)
    for ma, ta in enumerate(_HARMONICS[la]):
        for mb, tb in enumerate(_HARMONICS[lb]):
            for (ax, ay, az), fa in ta:
                for (bx, by, bz), fb in tb:
                    for t, ex in enumerate(e[0][(ax, bx)]):
                        for s, ey in enumerate(e[1][(ay, by)]):
                            for v, ez in enumerate(e[2][(az, bz)]):
                                u[:, herm[(t, s, v)], ma * (2 * lb + 1) + mb] += fa * fb * pref * ex * ey * ez
    aos = []
    for sa, sb in pairs:
        ia = [sh['ao_base'][sa] + m * sh['ao_stride'][sa] for m in range(2 * la + 1)]
        ib = [sh['ao_base'][sb] + m * sh['ao_stride'][sb] for m in range(2 * lb + 1)]
        aos.append([(x, y) for x in ia for y in ib])
    aos = torch.tensor(np.array(aos), device=device)
    return {'ltot': la + lb, 'n': len(pairs), 'owner': torch.tensor(owner, device=device), 'p': p, 'centre': centre,
            'u': u, 'ao_a': aos[:, :, 0], 'ao_b': aos[:, :, 1]}


def _class_block(bra, ket, omega2):
    """Contracted spherical integrals [bra pair, bra component, ket pair, ket component]."""
    top = bra['ltot'] + ket['ltot']
    nb, nk = bra['u'].shape[2], ket['u'].shape[2]
    hb, hk = _hermite_list(bra['ltot']), _hermite_list(ket['ltot'])
    hr = {h: i for i, h in enumerate(_hermite_list(top))}
    sign = torch.tensor([(-1.0) ** sum(q) for q in hk], dtype=torch.float64, device=bra['p'].device)
    uk = ket['u'] * sign[None, :, None]
    nkp = len(ket['p'])
    out = torch.zeros(bra['n'], nb, ket['n'], nk, dtype=torch.float64, device=bra['p'].device)
    step = max(1, _CHUNK // (nkp * max(len(hr) * 3, len(hb) * nk)))
    for s in range(0, len(bra['p']), step):
        p, pc = bra['p'][s:s + step, None], bra['centre'][s:s + step, None, :]
        q, qc = ket['p'][None, :], ket['centre'][None, :, :]
        rho = p * q / (p + q)
        scale = 2.0 * math.pi ** 2.5 / (p * q * torch.sqrt(p + q))
        if omega2 > 0.0:
            att = omega2 / (omega2 + rho)
            rho, scale = rho * att, scale * torch.sqrt(att)
        d = pc - qc
        boys = _boys(top, rho * (d * d).sum(-1))
        level = {}
        for n in range(top, -1, -1):
            new = {(0, 0, 0): scale * (-2.0 * rho) ** n * boys[n]}
            for h in _hermite_list(top - n)[1:]:
                x = next(k for k in range(3) if h[k] > 0)
                one = tuple(h[k] - (k == x) for k in range(3))
                v = d[..., x] * level[one]
                if h[x] > 1:
                    v = v + (h[x] - 1) * level[tuple(h[k] - 2 * (k == x) for k in range(3))]
                new[h] = v
            level = new
        r = torch.stack([level[h] for h in hr], dim=2)  # [bra primitives, ket primitives, hermite]
        del level, boys
        mid = torch.empty(r.shape[0], len(hb), nkp, nk, dtype=torch.float64, device=r.device)
        for i, h in enumerate(hb):
            at = torch.tensor([hr[tuple(h[k] + g[k] for k in range(3))] for g in hk], device=r.device)
            mid[:, i] = torch.bmm(r[:, :, at].permute(1, 0, 2).contiguous(), uk).permute(1, 0, 2)
        ub = bra['u'][s:s + step].permute(0, 2, 1).contiguous()
        prim = torch.bmm(ub, mid.reshape(mid.shape[0], len(hb), nkp * nk)).reshape(-1, nb, nkp, nk)
        half = torch.zeros(prim.shape[0], nb, ket['n'], nk, dtype=torch.float64, device=r.device)
        half.index_add_(2, ket['owner'], prim)
        out.index_add_(0, bra['owner'][s:s + step], half)
    return out


def _tensor(bas, mol, omega2):
    """All (pq|rs), n x n x n x n."""
    device = 'cuda:0' if torch.cuda.is_available() else 'cpu'
    sh = bas.shell_arrays(mol.get_coordinates_in_bohr())
    n = bas.get_dimensions_of_basis()
    lmax = int(max(sh['l']))
    sets = [_pair_class(sh, la, lb, device) for la in range(lmax + 1) for lb in range(la + 1)]
    sets = [s for s in sets if s is not None]
    eri = torch.zeros(n * n, n * n, dtype=torch.float64, device=device)
    for x, bra in enumerate(sets):
        for ket in sets[:x + 1]:
            blk = _class_block(bra, ket, omega2)
            m = blk.reshape(bra['n'] * blk.shape[1], ket['n'] * blk.shape[3])
            rows = [(bra['ao_a'] * n + bra['ao_b']).reshape(-1), (bra['ao_b'] * n + bra['ao_a']).reshape(-1)]
            cols = [(ket['ao_a'] * n + ket['ao_b']).reshape(-1), (ket['ao_b'] * n + ket['ao_a']).reshape(-1)]
            for r in rows:
                for c in cols:
                    eri[r[:, None], c[None, :]] = m
                    eri[c[:, None], r[None, :]] = m.T
    return eri, n


def _contract(eri, n, dens, fj, fk):
    """fj J + fk K of one density: J_pq = sum (pq|rs) D_rs, K_pr = sum (pq|rs) D_qs."""
    d = torch.from_numpy(dens).to(eri.device)
    out = torch.zeros(n, n, dtype=torch.float64, device=eri.device)
    if fj != 0.0:
        out += fj * (eri @ (0.5 * (d + d.T)).reshape(-1)).reshape(n, n)
    if fk != 0.0:
        cube = eri.reshape(n, n, n, n)
        for p in range(n):
            out[p] += fk * (cube[p].permute(1, 0, 2).reshape(n, n * n) @ d.reshape(-1))
    return out.cpu().numpy()


def _factors(label, xf):
    fj, fk, rs = LABELS[label]
    if fk is None:
        fk = -xf if label == '2jkx' else xf
    return fj, fk, rs


def exact(case, seed):
    kind = case['kind']
    if kind == 'train':
        return _exact_train(case, seed)
    if kind == 'batch':
        if case['molecules'] * case['most'] ** 2 > 100:
            return None
        got = []
        for mol, bas, d in _batch_molecules(case, seed):
            eri, n = _tensor(bas, mol, 0.0)
            fj, fk, _ = _factors(case['label'], 1.0)
            got.append(_contract(eri, n, d, fj, fk))
        return got
    mol, bas = _molecule(case, seed)
    if bas.get_dimensions_of_basis() > _EXACT_MOST:
        return None
    rng = np.random.Generator(np.random.PCG64(seed + 7))
    if kind == 'multi':
        eri, n = _tensor(bas, mol, 0.0)
        return [_contract(eri, n, d, *_factors(label, MULTI_XF)[:2])
                for label, _, d in _multi_densities(case, mol, bas, rng)]
    d = _density(mol, bas, rng)
    fj, fk, rs = _factors(case['label'], case['xf'])
    eri, n = _tensor(bas, mol, case['omega'] ** 2 if rs else 0.0)
    return _contract(eri, n, d, fj, fk)


def _exact_train(case, seed):
    """Loss and gradient of the SiLU network in float64."""
    x, t, shape, params = _train_inputs(case, seed)
    dims = ((N_IN, N_HIDDEN), (N_HIDDEN, N_HIDDEN), (N_HIDDEN, BLOCK * BLOCK))
    ws, at = [], 0
    for fi, fo in dims:
        ws.append(torch.tensor(params[at:at + fi * fo].reshape(fi, fo).astype(np.float64), requires_grad=True))
        at += fi * fo
        ws.append(torch.tensor(params[at:at + fo].astype(np.float64), requires_grad=True))
        at += fo
    h = torch.from_numpy(x.astype(np.float64))
    h = torch.nn.functional.silu(h @ ws[0] + ws[1])
    h = torch.nn.functional.silu(h @ ws[2] + ws[3])
    y = (h @ ws[4] + ws[5]).reshape(-1, BLOCK, BLOCK)
    s = torch.from_numpy(shape.astype(np.int64))
    at = torch.arange(BLOCK)
    mask = (at[None, :, None] < s[:, 0, None, None]) & (at[None, None, :] < s[:, 1, None, None])
    r = (y - torch.from_numpy(t.astype(np.float64)).reshape(-1, BLOCK, BLOCK)) * mask
    loss = ((r * r).sum((1, 2)) / (s[:, 0] * s[:, 1])).mean()
    loss.backward()
    return {'loss': float(loss.detach()), 'grad': torch.cat([w.grad.reshape(-1) for w in ws]).numpy()}
