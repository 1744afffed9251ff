"""The Boys-function table that every two-electron kernel reads, against the convergent series."""
import ctypes
import re

import numpy as np
import pytest

from veloxchem_amd import _native

NGRID, ROW, TMAX, LMAX = 289, 9, 36.0, 12


def _series(n, t):
    """F_n(t) = e^-t sum (2t)^k / ((2n+1) ... (2n+2k+1)), positive terms, in long double."""
    t = np.longdouble(t)
    term = np.longdouble(1) / (2 * n + 1)
    s = term
    for k in range(1, 400):
        term = term * 2 * t / (2 * n + 2 * k + 1)
        s += term
        if term < 1e-23 * s:
            break
    return np.exp(-t) * s


@pytest.mark.parametrize('L', [0, 1, 4, 6, 12])
def test_table_evaluation(L):
    """One table row (polynomial of degree 7, e^-T_k) and the downward recursion, at grid points, half-way
    between them and at the last point.  Each of the L + 1 steps rounds a few times: 4 + L eps."""
    if not _native.LIB_PATH.exists():
        pytest.skip('libvlxfock.so not built')
    lib = ctypes.CDLL(str(_native.LIB_PATH))
    build = getattr(lib, '_Z20vlx_build_boys_tablePd')
    build.restype = None
    tab = np.zeros((LMAX + 1, NGRID, ROW))
    build(tab.ctypes.data_as(ctypes.POINTER(ctypes.c_double)))
    src = (_native.LIB_PATH.parent / 'csrc' / 'vlx_boys.h').read_text()
    expd = [float(x) for x in re.search(r'BOYS_EXPD\[BOYS_ORDER \+ 1\] = \{([^}]*)\}', src).group(1).split(',')]
    T = np.r_[0.0, 1e-9, 0.0625, 0.06251, np.random.default_rng(0).uniform(0, TMAX, 200), TMAX - 0.0625, 35.99999]
    k = (T * 8 + 0.5).astype(int)
    d = T - k / 8
    c = tab[L][k]
    f, e = c[:, 7].copy(), np.full_like(d, expd[7])
    for j in range(6, -1, -1):
        f = f * d + c[:, j]
        e = e * d + expd[j]
    e *= c[:, 8]
    F = {L: f}
    for m in range(L - 1, -1, -1):
        F[m] = (2 * T * F[m + 1] + e) / (2 * m + 1)
    for m in range(L + 1):
        ref = np.array([float(_series(m, t)) for t in T])
        assert np.max(np.abs(F[m] - ref) / ref) <= (4 + L) * np.finfo(float).eps, m
