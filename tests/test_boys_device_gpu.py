"""The Boys function as the kernels evaluate it, through integrals that are one Hermite integral each."""
import ctypes

import numpy as np
import pytest

from tests.test_boys_table import _series
from veloxchem_amd import _native

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps
# the component of a shell that is a product of distinct coordinates: index, exponents, factor
PRODUCT = {0: (0, (0, 0, 0), 1.0), 1: (2, (1, 0, 0), 1.0), 2: (0, (1, 1, 0), 2.0 * np.sqrt(3.0)),
           3: (1, (1, 1, 1), 2.0 * np.sqrt(15.0))}


def _boys(top, args):
    got = np.empty((top + 1, len(args)), dtype=np.longdouble)
    for i, t in enumerate(args):
        if t <= 60.0:
            for m in range(top + 1):
                got[m, i] = _series(m, t)
        else:  # upward from F_0 = sqrt(pi / T) / 2, whose error erfc(sqrt(60)) is below 1e-26
            got[0, i] = np.sqrt(np.longdouble(np.pi) / t) / 2
            for m in range(top):
                got[m + 1, i] = ((2 * m + 1) * got[m, i] - np.exp(-t)) / (2 * t)
    return got


def _hermite(tuv, pq, rho, boys, n=0, absolute=False):
    """R^n_tuv of P - Q = pq; absolute: the sum of its terms' magnitudes."""
    if min(tuv) < 0:
        return 0.0
    x = next((k for k in range(3) if tuv[k] > 0), None)
    if x is None:
        r = (-2 * rho) ** n * boys[n]
        return abs(r) if absolute else r
    one, two = list(tuv), list(tuv)
    one[x] -= 1
    two[x] -= 2
    d = abs(pq[x]) if absolute else pq[x]
    return d * _hermite(tuple(one), pq, rho, boys, n + 1, absolute) + \
        (tuv[x] - 1) * _hermite(tuple(two), pq, rho, boys, n + 1, absolute)


@pytest.mark.parametrize('la, lc', [(0, 0), (1, 0), (1, 1), (2, 0), (2, 1), (2, 2), (3, 0), (3, 1), (3, 2), (3, 3)])
def test_device_boys_function(la, lc):
    """(la s|lc s), each pair on one centre, of the component that is a product of distinct coordinates:
    U R_{p+q} with one term.  Arguments at the middle between grid points, on them, next to the end of the
    table and past it.  A Boys value has 4 + L eps, and the argument's 6 eps move it by (L + 1/2) of that;
    a step of the recursion rounds three times, the prefactor eight times."""
    top = la + lc
    want = np.r_[0.0, 1e-10, 0.06249999, 0.06250001, 0.125, 1.0625, np.random.default_rng(la * 4 + lc).uniform(0, 36, 60),
                 35.874, 35.93749, 35.93751, 35.999999, 36.000001, 37.0, 80.0, 200.0]
    ea, ec, es = 0.8, 0.7, 0.9
    p, q = ea + es, ec + es
    rho = p * q / (p + q)
    way = np.array([1.0, 0.7, 0.4]) / np.linalg.norm([1.0, 0.7, 0.4])
    xyz = np.sqrt(want / rho)[:, None] * way
    k = len(want)
    ls = np.array([la, 0] + [lc, 0] * k, dtype=np.int32)
    ns = len(ls)
    centers = np.zeros((ns, 3))
    centers[2::2] = xyz
    centers[3::2] = xyz
    exps = np.array([ea, es] + [ec, es] * k)
    norms = np.ones(ns)
    width = 2 * ls + 1
    base = (np.cumsum(width) - width).astype(np.int32)
    one = np.ones(ns, dtype=np.int32)
    first = np.arange(ns, dtype=np.int32)
    lib, ctx = _native.lib(), _native.context()
    scr = ctypes.c_void_p()

    def ip(a):
        return a.ctypes.data_as(ctypes.POINTER(ctypes.c_int))

    def dp(a):
        return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    _native.check(lib.vlx_screener_create(ctx, ns, ip(ls), ip(one), ip(first), dp(exps), dp(norms),
                                          dp(np.ascontiguousarray(centers)), ip(base), ip(one), int(width.sum()),
                                          ctypes.byref(scr)))
    try:
        quartets = np.array([(0, 1, 2 + 2 * i, 3 + 2 * i) for i in range(k)], dtype=np.int32)
        out = np.zeros(k * (2 * la + 1) * (2 * lc + 1))
        _native.check(lib.vlx_eri_quartets(ctx, scr, k, ip(quartets), dp(out)))
    finally:
        lib.vlx_screener_destroy(scr)
    ia, ta, fa = PRODUCT[la]
    ic, tc, fc = PRODUCT[lc]
    got = out.reshape(k, 2 * la + 1, 2 * lc + 1)[:, ia, ic]
    pq = [-xyz[:, x].astype(np.longdouble) for x in range(3)]
    lrho = np.longdouble(p) * q / (np.longdouble(p) + q)
    boys = _boys(top, lrho * sum(d * d for d in pq))
    scale = 2 * np.longdouble(np.pi) ** 2.5 / (np.longdouble(p) * q * np.sqrt(np.longdouble(p) + q))
    scale = scale * fa * fc * (0.5 / np.longdouble(p)) ** la * (-0.5 / np.longdouble(q)) ** lc
    tuv = tuple(a + b for a, b in zip(ta, tc))
    ref = scale * _hermite(tuv, pq, lrho, boys)
    bound = (4 + top + 6 * (top + 0.5) + 3 * top + 8) * EPS * abs(scale) * _hermite(tuv, pq, lrho, boys, 0, True)
    assert np.all(np.abs(got - ref) <= bound), (want, np.asarray(np.abs(got - ref) / bound, dtype=float))
