// Boys-function table geometry (host and device).
#pragma once

// Grid T_k = k BOYS_DT, k < BOYS_NGRID, for T < BOYS_TMAX (larger T takes the asymptotic form).
// Row k of the table for L holds the BOYS_ORDER + 1 coefficients of the polynomial of degree
// BOYS_ORDER in d = T - T_k, |d| <= BOYS_DT / 2 = 1/16, that approximates F_L(T): the Taylor series
// around T_k with its terms above degree 7 economised by Chebyshev polynomials, absolute error below
// 3e-18 (the dropped Taylor term alone would be 3e-16), and then e^-T_k, from which
// e^-T = e^-T_k e^-d for the downward recursion (e^-d by BOYS_EXPD).
// Why this grid: the table is read from LDS at a row of its own in every lane, and these reads bound
// the low-L kernels.  Microbenchmark of one evaluation (16 waves per CU, random rows, CU cycles per
// wavefront): 22 doubles of row-major rows (order 10, spacing 1/4, F_L and F_{L-1}) 359; 8 doubles
// row-major with an odd stride 102; 8 doubles coefficient-major, the layout in LDS, 58.  Spacing
// 1/16 with degree 6 takes 52 but 32 KB instead of 20.3 KB.
constexpr int BOYS_ORDER = 7;
constexpr double BOYS_DT = 0.125;
constexpr double BOYS_INV_DT = 8.0;
constexpr int BOYS_NGRID = 289;
constexpr double BOYS_TMAX = 36.0;
constexpr int BOYS_EXP_COL = BOYS_ORDER + 1;  // column of e^-T_k
constexpr int BOYS_ROW = BOYS_ORDER + 2;
constexpr int BOYS_TAB_SIZE = BOYS_NGRID * BOYS_ROW;
constexpr int VLX_MAX_L = 3;
constexpr int VLX_MAX_LTOT = 4 * VLX_MAX_L;

// Coefficients of e^-d, |d| <= 1/16: the same economised polynomial of degree 7 (error below 6e-17).
constexpr double BOYS_EXPD[BOYS_ORDER + 1] = {
    1.0, -1.0, 0.5000000000003696, -0.16666666666674368,
    0.04166666619357543, -0.00833333326237029, 0.0013890826631164288, -0.00019843692002687578};

// Fills tab[(L * BOYS_NGRID + k) * BOYS_ROW + j] (row-major) for L = 0..VLX_MAX_LTOT.
void vlx_build_boys_table(double* tab);
