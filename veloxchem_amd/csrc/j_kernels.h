// Coulomb builds without exchange (labels "j" and "j_rs"): J through Hermite densities.
//
//   J_ab = sum_prim sum_p U_ab[p] J_p,   J_p = sum_ket prims sum_q R_{p+q} H_q,
//   H_q = (-1)^q sum_cd U_cd[q] D_cd
//
// with U the Hermite-to-spherical matrix of a primitive pair.  H is made once per primitive of every
// pair (j_engine.hip) and U_ab is applied once at the end, so a primitive quartet costs its Boys function,
// the recursion to R^0 and one product per (p, q): no horizontal recursion, no integrals, no digestion.
// The class kernels spend 70-90% of a Coulomb build on those.  Every primitive of one Hermite rank
// (la + lb) is in one list, whatever its pair class, sorted by the pair's Schwarz bin, so that the pair
// screening of the class kernels (bin_bra + bin_ket <= ithreshold) is again a prefix of the list.
// Both orders of a quartet are visited: half the recursions could be saved by adding to the ket's J_q as
// well, but every lane would then reduce or scatter that sum for each ket.
//
// Bound by the FP64 vector units, busy 84 to 94% of the time in the launches of ranks up to 3: a lane
// keeps one bra primitive, its J_p and R^0 in registers, the kets pass through LDS as broadcasts.  The
// ranks above it are held to 4 waves a CU by their registers, at 36 to 67%.  27 waters def2-TZVP, label
// j: 116 ms with the class kernels, 32 ms so; run one after another the largest launches are those of the
// lowest ranks, (1,0), (0,1), (1,1) and (0,0) at 2.0 to 2.4 ms of 29, beside 9 ms of class kernels.
#pragma once

#include "eri_kernels.h"
#include "vlx_jtypes.h"

// Hermite functions of degree <= N in order of degree: exponents, and for the recursion
// R_{t+1} = x R_t + t R_{t-1} the axis and the indices of the two lower functions.
template <int N>
struct JHerm {
    int t[j_nherm(N)], u[j_nherm(N)], v[j_nherm(N)];
    int axis[j_nherm(N)], lo1[j_nherm(N)], lo2[j_nherm(N)], fac[j_nherm(N)];
};
constexpr int j_index(int t, int u, int v)
{
    const int n = t + u + v;
    // degree n: t from n down, u from n - t down
    const int before = (n - t) * (n - t + 1) / 2;
    return j_nherm(n - 1) + before + (n - t - u);
}
template <int N>
constexpr JHerm<N> j_make()
{
    JHerm<N> h{};
    for (int n = 0; n <= N; n++)
        for (int t = n; t >= 0; t--)
            for (int u = n - t; u >= 0; u--) {
                const int v = n - t - u, i = j_index(t, u, v);
                h.t[i] = t, h.u[i] = u, h.v[i] = v;
                if (n == 0) continue;
                // an axis of exponent 1 needs no second term
                const int ax = t == 1 ? 0 : u == 1 ? 1 : v == 1 ? 2 : t > 0 ? 0 : u > 0 ? 1 : 2;
                const int e = ax == 0 ? t : ax == 1 ? u : v;
                h.axis[i] = ax;
                h.fac[i] = e - 1;
                h.lo1[i] = j_index(t - (ax == 0), u - (ax == 1), v - (ax == 2));
                h.lo2[i] = e > 1 ? j_index(t - 2 * (ax == 0), u - 2 * (ax == 1), v - 2 * (ax == 2)) : 0;
            }
    return h;
}

// kets of a stage of the LDS pipeline
constexpr int j_stage(int lcd) { return lcd <= 2 ? 64 : 32; }

template <int LAB, int LCD, bool RS>
__global__ void __launch_bounds__(JBLOCK) j_kernel(const JArgs a)
{
    constexpr int L = LAB + LCD, NH = j_nherm(LAB), NK = j_nherm(LCD), NR = j_nherm(L), ROW = j_row(LCD);
    constexpr int STAGE = j_stage(LCD);
    constexpr JHerm<L> h = j_make<L>();
    __shared__ double tab[BOYS_TAB_SIZE];
    __shared__ double kets[STAGE * ROW];
    stage_boys(tab, a.boys_tab);
    for (int it = blockIdx.x; it < a.nitems; it += gridDim.x) {
        const JItem ji = a.items[it];
        const int e = ji.i0 + static_cast<int>(threadIdx.x);
        const bool in = e < a.nbra;
        const double* bp = a.bra + (size_t)min(e, a.nbra - 1) * j_row(LAB);
        const double zeta = bp[0], px = bp[1], py = bp[2], pz = bp[3];
        // kets the lane's bra meets: a prefix of the list
        const int lim = a.ithreshold - a.bra_bin[min(e, a.nbra - 1)];
        const int kend = in && lim >= 0 ? min(ji.k1, a.ket_cnt[min(lim, 15)]) : 0;
        double acc[NH];
#pragma unroll
        for (int p = 0; p < NH; p++) acc[p] = 0.0;
        for (int s0 = ji.k0; s0 < ji.k1; s0 += STAGE) {
            const int ns = min(STAGE, ji.k1 - s0);
            __syncthreads();
            for (int i = threadIdx.x; i < ns * ROW; i += JBLOCK) kets[i] = a.ket[(size_t)s0 * ROW + i];
            __syncthreads();
            const int mine = min(ns, kend - s0);
            for (int k = 0; k < mine; k++) {
                const double* kp = kets + k * ROW;
                const double sz = zeta + kp[0];
                const double rho_c = zeta * kp[0] * vrcp<double>(sz);
                double rho = rho_c, w = vrsqrt<double>(sz);
                if constexpr (RS) {
                    const double sfac = a.omega2 / (a.omega2 + rho_c);
                    rho = rho_c * sfac;
                    w *= sqrt(sfac);
                }
                const double pq[3] = {px - kp[1], py - kp[2], pz - kp[3]};
                double seed[L + 1];
                boys_eval<L, double>(rho * (pq[0] * pq[0] + pq[1] * pq[1] + pq[2] * pq[2]), tab, seed);
#pragma unroll
                for (int n = 0; n <= L; n++) {
                    seed[n] *= w;
                    w *= -2.0 * rho;
                }
                // R^n from R^{n+1} in place, highest degree first
                double r[NR];
                r[0] = seed[L];
#pragma unroll
                for (int n = L - 1; n >= 0; n--) {
#pragma unroll
                    for (int i = NR - 1; i >= 1; i--) {
                        if (i < j_nherm(L - n)) {
                            const double x = pq[h.axis[i]] * r[h.lo1[i]];
                            r[i] = h.fac[i] > 0 ? fma(static_cast<double>(h.fac[i]), r[h.lo2[i]], x) : x;
                        }
                    }
                    r[0] = seed[n];
                }
#pragma unroll
                for (int q = 0; q < NK; q++) {
                    const double hq = kp[4 + q];
#pragma unroll
                    for (int p = 0; p < NH; p++)
                        acc[p] = fma(r[j_index(h.t[p] + h.t[q], h.u[p] + h.u[q], h.v[p] + h.v[q])], hq, acc[p]);
                }
            }
        }
        if (kend > ji.k0) {
#pragma unroll
            for (int p = 0; p < NH; p++) unsafeAtomicAdd(a.jp + (size_t)e * NH + p, acc[p]);
        }
    }
}
