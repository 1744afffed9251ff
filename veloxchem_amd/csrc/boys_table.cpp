// Host generation of the Boys-function table used by the kernels.
//
// F_n(T) = integral_0^1 t^(2n) exp(-T t^2) dt is evaluated in long double
// (64-bit mantissa) from the convergent series
//   F_n(T) = exp(-T) sum_{k>=0} (2T)^k / ((2n+1)(2n+3)...(2n+2k+1)),
// whose terms are all positive (no cancellation), so each table entry is
// accurate to well below double rounding.  The reference tabulates the same
// function (src/math/BoysFunc.hpp:24806-24888); this table is generated here
// from the definition, with its own grid spacing and order.
#include <cmath>
#include <cstddef>

#include "vlx_boys.h"

// Taylor terms kept before the economisation: (1/16)^17 / 17! is far below long double rounding.
constexpr int BOYS_TAYLOR = 16;

static long double boys_series(int n, long double t)
{
    long double term = 1.0L / (2 * n + 1);
    long double sum = term;
    for (int k = 1; k < 2000; k++) {
        term *= 2.0L * t / (2 * n + 2 * k + 1);
        sum += term;
        if (term < 1.0e-22L * sum) break;
    }
    return expl(-t) * sum;
}

// Coefficients of the Chebyshev polynomial T_n in powers of x.
static void chebyshev(int n, long double* c)
{
    long double a[BOYS_TAYLOR + 1] = {1.0L}, b[BOYS_TAYLOR + 1] = {0.0L, 1.0L};
    for (int i = 0; i <= BOYS_TAYLOR; i++) c[i] = (n == 0) ? a[i] : b[i];
    for (int m = 2; m <= n; m++) {
        for (int i = 0; i <= BOYS_TAYLOR; i++) c[i] = (i > 0 ? 2.0L * b[i - 1] : 0.0L) - a[i];
        for (int i = 0; i <= BOYS_TAYLOR; i++) {
            a[i] = b[i];
            b[i] = c[i];
        }
    }
}

void vlx_build_boys_table(double* tab)
{
    constexpr int nmax = VLX_MAX_LTOT + BOYS_TAYLOR;
    const long double h = 0.5L * BOYS_DT;
    static long double f[BOYS_NGRID][nmax + 1];
    long double cheb[BOYS_TAYLOR + 1][BOYS_TAYLOR + 1];
    for (int n = 0; n <= BOYS_TAYLOR; n++) chebyshev(n, cheb[n]);
    for (int k = 0; k < BOYS_NGRID; k++)
        for (int n = 0; n <= nmax; n++) f[k][n] = boys_series(n, (long double)k * BOYS_DT);
    for (int L = 0; L <= VLX_MAX_LTOT; L++)
        for (int k = 0; k < BOYS_NGRID; k++) {
            // Taylor series of F_L around T_k in x = d / h, |x| <= 1: F_L^(j) = (-1)^j F_{L+j}
            long double b[BOYS_TAYLOR + 1], scale = 1.0L;
            for (int j = 0; j <= BOYS_TAYLOR; j++) {
                if (j > 0) scale *= -h / j;
                b[j] = f[k][L + j] * scale;
            }
            // the terms above BOYS_ORDER, from the top, as multiples of T_n moved to the lower powers
            for (int n = BOYS_TAYLOR; n > BOYS_ORDER; n--) {
                const long double m = b[n] / cheb[n][n];
                for (int i = 0; i <= n; i++) b[i] -= m * cheb[n][i];
            }
            double* row = tab + (size_t)(L * BOYS_NGRID + k) * BOYS_ROW;
            long double hj = 1.0L;
            for (int j = 0; j <= BOYS_ORDER; j++, hj *= h) row[j] = (double)(b[j] / hj);
            row[BOYS_EXP_COL] = (double)expl(-(long double)k * BOYS_DT);
        }
}
