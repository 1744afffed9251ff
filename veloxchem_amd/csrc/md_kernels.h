// Wavefront-cooperative electron-repulsion kernels for the largest classes
// (f shells), where straight-line recursions would neither fit the register
// file nor compile in reasonable time.
//
// One shell quartet at a time per wavefront (work-group = one wavefront),
// McMurchie-Davidson in matrix form, everything staged in LDS:
//   U_AB[ab][p]  = k_ab sum_{cart a,b} S_a S_b E^{ab,x}_t E^{ab,y}_u E^{ab,z}_v
//                  (Hermite expansion of a bra primitive pair projected on the
//                   real solid harmonics of src/general/SphericalMomentum.hpp)
//   R[n][tuv]    = Hermite Coulomb integrals, by the recursion
//                  R^n_{t+1,u,v} = t R^{n+1}_{t-1,u,v} + X_PQ R^{n+1}_{t,u,v}
//                  from R^n_000 = (-2 rho)^n F_n(rho |PQ|^2)
//   X[p][cd]     = sum_q R[p+q] (-1)^{|q|} U_CD[cd][q]
//   out[ab][cd] += sum_p U_AB[ab][p] X[p][cd] / sqrt(zeta + eta)
// with lanes parallel over matrix entries.  The spherical block in LDS is
// then digested (Fock), stored (explicit quartets) or reduced (screener).
#pragma once

#include <algorithm>

#include "eri_kernels.h"

namespace md {

constexpr int nherm(int l) { return (l + 1) * (l + 2) * (l + 3) / 6; }
constexpr int D1 = VLX_MAX_L + 1;
constexpr int DT = 2 * VLX_MAX_L + 1;
constexpr int E3 = D1 * D1 * DT;  // 1D coefficients per axis; an E array holds 3 axes

// linear index of Hermite (t,u,v): degree-major, then (t descending, u descending)
__device__ __forceinline__ int hidx(int t, int u, int v)
{
    const int n = t + u + v, s = u + v;
    return n * (n + 1) * (n + 2) / 6 + s * (s + 1) / 2 + v;
}

__device__ __forceinline__ void hdecode(int idx, int& t, int& u, int& v)
{
    int n = 0;
    while (nherm(n) <= idx) n++;
    const int rem = idx - (n > 0 ? nherm(n - 1) : 0);
    int s = 0;
    while ((s + 1) * (s + 2) / 2 <= rem) s++;
    v = rem - s * (s + 1) / 2;
    u = s - v;
    t = n - s;
}

// Cartesian exponents of component c of shell l (xx, xy, xz, yy, yz, zz, ...)
__device__ __forceinline__ void cart_exp(int l, int c, int& x, int& y, int& z)
{
    int i = 0;
    for (int xx = l; xx >= 0; xx--)
        for (int yy = l - xx; yy >= 0; yy--, i++)
            if (i == c) {
                x = xx;
                y = yy;
                z = l - xx - yy;
                return;
            }
    x = y = z = 0;
}

// Spherical component m of shell l as Cartesian terms (index, factor); the
// factors and orders are those of src/general/SphericalMomentum.hpp:18-134.
__device__ __forceinline__ int sph_terms(int l, int m, int* ci, double* cf)
{
    const double f3 = 3.46410161513775458705;   // 2 sqrt(3)
    const double g5 = 1.58113883008418966599;   // sqrt(5/2)
    const double g15 = 7.74596669241483377036;  // 2 sqrt(15)
    const double g3 = 1.22474487139158904910;   // sqrt(3/2)
    switch (l * 8 + m) {
    case 0: ci[0] = 0; cf[0] = 1.0; return 1;
    case 8: ci[0] = 1; cf[0] = 1.0; return 1;
    case 9: ci[0] = 2; cf[0] = 1.0; return 1;
    case 10: ci[0] = 0; cf[0] = 1.0; return 1;
    case 16: ci[0] = 1; cf[0] = f3; return 1;
    case 17: ci[0] = 4; cf[0] = f3; return 1;
    case 18: ci[0] = 0; cf[0] = -1.0; ci[1] = 3; cf[1] = -1.0; ci[2] = 5; cf[2] = 2.0; return 3;
    case 19: ci[0] = 2; cf[0] = f3; return 1;
    case 20: ci[0] = 0; cf[0] = 0.5 * f3; ci[1] = 3; cf[1] = -0.5 * f3; return 2;
    case 24: ci[0] = 1; cf[0] = 3.0 * g5; ci[1] = 6; cf[1] = -g5; return 2;
    case 25: ci[0] = 4; cf[0] = g15; return 1;
    case 26: ci[0] = 8; cf[0] = 4.0 * g3; ci[1] = 1; cf[1] = -g3; ci[2] = 6; cf[2] = -g3; return 3;
    case 27: ci[0] = 9; cf[0] = 2.0; ci[1] = 2; cf[1] = -3.0; ci[2] = 7; cf[2] = -3.0; return 3;
    case 28: ci[0] = 5; cf[0] = 4.0 * g3; ci[1] = 0; cf[1] = -g3; ci[2] = 3; cf[2] = -g3; return 3;
    case 29: ci[0] = 2; cf[0] = 0.5 * g15; ci[1] = 7; cf[1] = -0.5 * g15; return 2;
    case 30: ci[0] = 0; cf[0] = g5; ci[1] = 3; cf[1] = -3.0 * g5; return 2;
    default: return 0;
    }
}

template <int la, int lb, int lc, int ld>
struct Sizes {
    static constexpr int L = la + lb + lc + ld;
    static constexpr int nhab = nherm(la + lb), nhcd = nherm(lc + ld), nr = nherm(L);
    static constexpr int nsa = 2 * la + 1, nsb = 2 * lb + 1, nsc = 2 * lc + 1, nsd = 2 * ld + 1;
    static constexpr int nsab = nsa * nsb, nscd = nsc * nsd;
    // LDS doubles: E (bra, ket), U_AB, U_CD, two R levels, X, out, scalars
    static constexpr int lds = 6 * E3 + nsab * nhab + nhcd * nscd + 2 * nr + nhab * nscd + nsab * nscd + 32;
    // the Boys table is staged in LDS when it fits beside the work arrays, else read from HBM/L2
    static constexpr bool tab_in_lds = (lds + nsab * nscd + BOYS_TAB_SIZE) * 8 <= 160 * 1024;
};

// 1D Hermite coefficients E^{ij}_t (i <= la, j <= lb) of one primitive pair for
// axis x = threadIdx.x < 3; pa = P - A, pb = P - B.
__device__ __forceinline__ void hermite_1d(int la, int lb, double p, const double* pa, const double* pb,
                                           double* __restrict__ e)
{
    const int x = threadIdx.x;
    if (x >= 3) return;
    double* ex = e + x * E3;
    for (int k = 0; k < E3; k++) ex[k] = 0.0;
    const double h = 0.5 / p;
    ex[0] = 1.0;
    for (int i = 0; i <= la; i++)
        for (int j = 0; j <= lb; j++) {
            if (i == 0 && j == 0) continue;
            for (int t = 0; t <= i + j; t++) {
                double v;
                if (j == 0) {
                    const double* src = ex + ((i - 1) * D1 + j) * DT;
                    v = pa[x] * src[t];
                    if (t > 0) v += h * src[t - 1];
                    if (t + 1 <= i - 1 + j) v += (t + 1) * src[t + 1];
                } else {
                    const double* src = ex + (i * D1 + (j - 1)) * DT;
                    v = pb[x] * src[t];
                    if (t > 0) v += h * src[t - 1];
                    if (t + 1 <= i + j - 1) v += (t + 1) * src[t + 1];
                }
                ex[(i * D1 + j) * DT + t] = v;
            }
        }
}

// Bra: u[ab * nh + p]; ket (sign (-1)^{t+u+v}): u[p * ns + cd]; scaled by k.
__device__ __forceinline__ void build_u(int la, int lb, const double* __restrict__ e, double k, bool ket,
                                        double* __restrict__ u)
{
    const int nsb = 2 * lb + 1, ns = (2 * la + 1) * nsb, nh = nherm(la + lb);
    for (int idx = threadIdx.x; idx < ns * nh; idx += blockDim.x) {
        const int ab = idx / nh, ph = idx % nh;
        int t, uu, v;
        hdecode(ph, t, uu, v);
        int cia[3], cib[3];
        double cfa[3], cfb[3];
        const int nta = sph_terms(la, ab / nsb, cia, cfa);
        const int ntb = sph_terms(lb, ab % nsb, cib, cfb);
        double acc = 0.0;
        for (int ia = 0; ia < nta; ia++) {
            int ax, ay, az;
            cart_exp(la, cia[ia], ax, ay, az);
            for (int ib = 0; ib < ntb; ib++) {
                int bx, by, bz;
                cart_exp(lb, cib[ib], bx, by, bz);
                if (t > ax + bx || uu > ay + by || v > az + bz) continue;
                acc += cfa[ia] * cfb[ib] * e[(ax * D1 + bx) * DT + t] * e[E3 + (ay * D1 + by) * DT + uu] *
                       e[2 * E3 + (az * D1 + bz) * DT + v];
            }
        }
        if (ket) {
            if ((t + uu + v) & 1) acc = -acc;
            u[ph * ns + ab] = k * acc;
        } else {
            u[ab * nh + ph] = k * acc;
        }
    }
}

// Cooperative spherical block (ab|cd) -> out[ab * nscd + cd] in LDS.
// ab_vec = A - B, cd_vec = C - D (P - B = (P - A) + (A - B)).
template <int la, int lb, int lc, int ld>
__device__ void quartet(const PrimPair* __restrict__ bra_prims, int bra_np, const double* ab_vec,
                        const PrimPair* __restrict__ ket_prims, int ket_np, const double* cd_vec,
                        const double* __restrict__ tab, const double omega2, double* __restrict__ lds,
                        double* __restrict__ out)
{
    using S = Sizes<la, lb, lc, ld>;
    constexpr int L = S::L;
    double* ebra = lds;
    double* eket = ebra + 3 * E3;
    double* uab = eket + 3 * E3;
    double* ucd = uab + S::nsab * S::nhab;
    double* ra = ucd + S::nhcd * S::nscd;
    double* rb = ra + S::nr;
    double* x = rb + S::nr;
    double* scal = x + S::nhab * S::nscd;  // Boys values F_0..F_L
    for (int k = threadIdx.x; k < S::nsab * S::nscd; k += blockDim.x) out[k] = 0.0;
    for (int ib = 0; ib < bra_np; ib++) {
        const PrimPair bp = bra_prims[ib];
        {
            const double pa[3] = {bp.pax, bp.pay, bp.paz};
            const double pb[3] = {bp.pax + ab_vec[0], bp.pay + ab_vec[1], bp.paz + ab_vec[2]};
            __syncthreads();
            hermite_1d(la, lb, bp.zeta, pa, pb, ebra);
            __syncthreads();
            build_u(la, lb, ebra, bp.k, false, uab);
        }
        for (int ik = 0; ik < ket_np; ik++) {
            const PrimPair kp = ket_prims[ik];
            const double qc[3] = {kp.pax, kp.pay, kp.paz};
            const double qd[3] = {kp.pax + cd_vec[0], kp.pay + cd_vec[1], kp.paz + cd_vec[2]};
            __syncthreads();
            hermite_1d(lc, ld, kp.zeta, qc, qd, eket);
            const double s = bp.zeta + kp.zeta;
            // erf(omega r)/r: rho -> sfac rho and a factor sqrt(sfac), sfac = omega^2 / (omega^2 + rho)
            const double rho_c = bp.zeta * kp.zeta / s;
            const double sfac = (omega2 > 0.0) ? omega2 / (omega2 + rho_c) : 1.0;
            const double rho = (omega2 > 0.0) ? rho_c * sfac : rho_c;
            const double pq[3] = {bp.px - kp.px, bp.py - kp.py, bp.pz - kp.pz};
            if (threadIdx.x == 3) {
                double F[L + 1];
                boys_eval<L, double, true>(rho * (pq[0] * pq[0] + pq[1] * pq[1] + pq[2] * pq[2]), tab, F);
                for (int m = 0; m <= L; m++) scal[m] = F[m];
            }
            __syncthreads();
            build_u(lc, ld, eket, kp.k, true, ucd);
            // R levels n = L .. 0 (ping-pong between ra and rb)
            double* cur = (L & 1) ? rb : ra;
            if (threadIdx.x == 0) {
                double f = 1.0;
                for (int m = 0; m < L; m++) f *= -2.0 * rho;
                cur[0] = f * scal[L];
            }
            for (int n = L - 1; n >= 0; n--) {
                double* prev = cur;
                cur = (cur == ra) ? rb : ra;
                __syncthreads();
                double fn = 1.0;
                for (int m = 0; m < n; m++) fn *= -2.0 * rho;
                for (int idx = threadIdx.x; idx < nherm(L - n); idx += blockDim.x) {
                    int t, u, v;
                    hdecode(idx, t, u, v);
                    double val;
                    if (t > 0) {
                        val = pq[0] * prev[hidx(t - 1, u, v)];
                        if (t > 1) val += (t - 1) * prev[hidx(t - 2, u, v)];
                    } else if (u > 0) {
                        val = pq[1] * prev[hidx(t, u - 1, v)];
                        if (u > 1) val += (u - 1) * prev[hidx(t, u - 2, v)];
                    } else if (v > 0) {
                        val = pq[2] * prev[hidx(t, u, v - 1)];
                        if (v > 1) val += (v - 1) * prev[hidx(t, u, v - 2)];
                    } else {
                        val = fn * scal[n];
                    }
                    cur[idx] = val;
                }
            }
            __syncthreads();
            // X[p][cd] = sum_q R[p+q] U_CD[q][cd]
            for (int idx = threadIdx.x; idx < S::nhab * S::nscd; idx += blockDim.x) {
                const int p = idx / S::nscd, cd = idx % S::nscd;
                int t, u, v;
                hdecode(p, t, u, v);
                double acc = 0.0;
                for (int q = 0; q < S::nhcd; q++) {
                    int tq, uq, vq;
                    hdecode(q, tq, uq, vq);
                    acc = fma(cur[hidx(t + tq, u + uq, v + vq)], ucd[q * S::nscd + cd], acc);
                }
                x[idx] = acc;
            }
            __syncthreads();
            const double w = (omega2 > 0.0) ? sqrt(sfac) / sqrt(s) : 1.0 / sqrt(s);
            for (int idx = threadIdx.x; idx < S::nsab * S::nscd; idx += blockDim.x) {
                const int ab = idx / S::nscd, cd = idx % S::nscd;
                double acc = 0.0;
                for (int p = 0; p < S::nhab; p++) acc = fma(uab[ab * S::nhab + p], x[p * S::nscd + cd], acc);
                out[idx] += w * acc;
            }
        }
    }
    __syncthreads();
}

}  // namespace md

// ------------------------------------------------------------------------
// Matrix-core McMurchie-Davidson Fock kernel.
//
// The Hermite-to-spherical matrices of every primitive pair are built once
// per screener (u_build_kernel) and stored in HBM as
//   U[prim][h][s] = k sum_{cart a, b} S_a S_b E^x E^y E^z
// (h < nherm(la + lb) Hermite index, s < (2la+1)(2lb+1) spherical index, both
// padded to multiples of 16 with zeros; a ket's U carries the sign (-1)^|h|).  One
// wavefront takes one shell quartet at a time; per primitive quartet it builds
// R^0[tuv] (scaled by 1/sqrt(zeta + eta)) in LDS and runs two FP64 matrix-core products
//   X[p][cd]    = sum_q R^0[p + q] U_CD[q][cd]                   (v_mfma_f64_16x16x4)
//   out[ab][cd] += sum_p U_AB[p][ab] X[p][cd]
// Operand layouts of v_mfma_f64_16x16x4f64 (wave64): A[i][k] in lane i + 16k, B[k][j] in lane
// j + 16k, D[i][j] in register i / 4 of lane j + 16 (i % 4).  So register r of X's row tile m is, in
// every lane, the B operand of the second product's step 4m + r: X never leaves the registers.  The
// byte offset of R^0[p + q] of every step of the first product is a constant of the lane, computed
// once per wavefront and kept packed in registers, as are the steps of the R recursion and the
// operands of the digestion.
//
// Digestion: the six F' blocks' elements, each with the D block it contracts, are dealt to the lanes
// in order of their number of terms (146 elements in three rounds of 35, 21 and 15 terms for (fd|dp)),
// instead of one block after another with 15 to 35 of 64 lanes at work.  An element's F' address is
// also the address of the D element that the lane fetches, at the quartet's start, behind the
// integrals.

using md::hidx;
using md::nherm;

struct HermDecode {
    int e[nherm(VLX_MAX_LTOT)];  // t | u << 8 | v << 16 of Hermite index idx
};
constexpr HermDecode make_herm_decode()
{
    HermDecode d{};
    int i = 0;
    for (int n = 0; n <= VLX_MAX_LTOT; n++)
        for (int s = 0; s <= n; s++)
            for (int v = 0; v <= s; v++) d.e[i++] = (n - s) | ((s - v) << 8) | (v << 16);
    return d;
}
static __device__ constexpr HermDecode g_herm = make_herm_decode();

// The step of the R recursion that produces Hermite index idx (t, u, v), as one packed int:
// s1 | s2 << 9 | axis << 18 | c << 20.  Along the first axis with a nonzero index (x for t > 0,
// else y, else z; k the index along it), R^n[idx] = PQ_axis R^{n+1}[s1] + c R^{n+1}[s2] with
// s1 the index one lower along the axis, s2 two lower and c = k - 1 (s2 = 0 and c = 0 for k = 1;
// idx 0 takes the seed).  Indices stay below 2^9 (nherm(VLX_MAX_LTOT) = 455).
struct HermRecur {
    int e[nherm(VLX_MAX_LTOT)];
};
constexpr HermRecur make_herm_recur()
{
    HermRecur r{};
    auto lin = [](int t, int u, int v) {
        const int n = t + u + v, s = u + v;
        return n * (n + 1) * (n + 2) / 6 + s * (s + 1) / 2 + v;
    };
    int i = 0;
    for (int n = 0; n <= VLX_MAX_LTOT; n++)
        for (int s = 0; s <= n; s++)
            for (int v = 0; v <= s; v++) {
                const int t = n - s, u = s - v;
                int s1 = 0, s2 = 0, axis = 0, c = 0;
                if (t > 0) {
                    s1 = lin(t - 1, u, v);
                    if (t > 1) s2 = lin(t - 2, u, v), c = t - 1;
                } else if (u > 0) {
                    axis = 1;
                    s1 = lin(t, u - 1, v);
                    if (u > 1) s2 = lin(t, u - 2, v), c = u - 1;
                } else if (v > 0) {
                    axis = 2;
                    s1 = lin(t, u, v - 1);
                    if (v > 1) s2 = lin(t, u, v - 2), c = v - 1;
                }
                r.e[i++] = s1 | (s2 << 9) | (axis << 18) | (c << 20);
            }
    return r;
}
static __device__ constexpr HermRecur g_hrec = make_herm_recur();
static_assert(nherm(VLX_MAX_LTOT) <= 512, "R recursion table packs indices in 9 bits");

__device__ __forceinline__ int hidx_packed(int tuv)
{
    return hidx(tuv & 0xff, (tuv >> 8) & 0xff, tuv >> 16);
}

typedef double vlx_d4 __attribute__((ext_vector_type(4)));

template <int la, int lb, int lc, int ld>
struct MmdSizes {
    static constexpr int L = la + lb + lc + ld;
    static constexpr int nhab = nherm(la + lb), nhcd = nherm(lc + ld), nr = nherm(L);
    static constexpr int na = 2 * la + 1, nb = 2 * lb + 1, nc = 2 * lc + 1, nd = 2 * ld + 1;
    static constexpr int nsab = na * nb, nscd = nc * nd;
    static constexpr int HA = vlx_u_rows(la, lb), SA = vlx_u_cols(la, lb);  // bra U: HA x SA
    static constexpr int HC = vlx_u_rows(lc, ld), SC = vlx_u_cols(lc, ld);  // ket U: HC x SC
    static constexpr int MT = SA / 16, NT = SC / 16, MX = (nhab + 15) / 16;
    static constexpr int KX = (nhcd + 3) / 4, KO = (nhab + 3) / 4;
    static constexpr int KR = (nr + VLX_WAVE - 1) / VLX_WAVE;  // entries of R^0 per lane
    // X summed over the ket primitives before the second product, where its tiles fit in registers
    static constexpr bool XSUM = MX * NT <= 6;
    // U_CD operands of a primitive quartet fetched ahead of the R recursion
    static constexpr bool PRE_X = KX * NT <= 12;
    // elements of the six blocks AB, CD, AC, AD, BC, BD and rounds of the digestion
    static constexpr int nout = nsab + nscd + (na + nb) * (nc + nd);
    static constexpr int NR = (nout + VLX_WAVE - 1) / VLX_WAVE;
    // estimated VGPRs, for the occupancy the registers are held to
    static constexpr int regs = 8 * MT * NT + 8 * MX * (XSUM ? NT : 1) + MX * KX / 2 + 5 * KR + 2 * (L + 1) + 8 * NR +
                                (PRE_X ? 2 * KX * NT : 8) + 40;
    static constexpr int occupancy = regs <= 128 ? 4 : regs <= 170 ? 3 : regs <= 256 ? 2 : 1;
};

// Digestion of one shell quartet over the lanes: element o (in order of decreasing term count) of the
// six blocks.  Element (x, y) of block X sums I[..] over the elements (u, v) of its partner block
// (AB with CD, AC with BD, AD with BC): I offset x sx + y sy + u su + v sv, partner element u nv + v.
template <int la, int lb, int lc, int ld>
struct MmdDigest {
    using S = MmdSizes<la, lb, lc, ld>;
    struct Tab {
        int ib[S::nout];     // byte offset of the first integral | of the partner block in LDS << 16
        int step[S::nout];   // byte step of v | steps of v per u << 16 | terms << 24
        int wrap[S::nout];   // extra byte step after nv steps | LDS slot of the element's D << 16
        int addr[S::nout];   // row shell | row component << 2 | column shell << 5 | column component << 7 | Coulomb << 10
        int terms[S::NR];    // most terms of a round
    };
    static constexpr Tab make()
    {
        Tab t{};
        constexpr int n[4] = {S::na, S::nb, S::nc, S::nd};
        constexpr int st[4] = {S::nb * S::nc * S::nd, S::nc * S::nd, S::nd, 1};
        constexpr int blk[6][2] = {{0, 1}, {2, 3}, {0, 2}, {0, 3}, {1, 2}, {1, 3}};
        constexpr int partner[6] = {1, 0, 5, 4, 3, 2};
        int base[6] = {}, used[6] = {};
        for (int b = 1; b < 6; b++) base[b] = base[b - 1] + n[blk[b - 1][0]] * n[blk[b - 1][1]];
        int o = 0;
        for (int k = 0; k < 6; k++) {
            int best = -1, most = -1;
            for (int b = 0; b < 6; b++) {
                const int terms = n[blk[partner[b]][0]] * n[blk[partner[b]][1]];
                if (!used[b] && terms > most) best = b, most = terms;
            }
            used[best] = 1;
            const int x = blk[best][0], y = blk[best][1], u = blk[partner[best]][0], v = blk[partner[best]][1];
            for (int i = 0; i < n[x]; i++)
                for (int j = 0; j < n[y]; j++, o++) {
                    t.ib[o] = 8 * (i * st[x] + j * st[y]) | (8 * base[partner[best]]) << 16;
                    t.step[o] = 8 * st[v] | n[v] << 16 | most << 24;
                    t.wrap[o] = 8 * (st[u] - n[v] * st[v]) | (base[best] + i * n[y] + j) << 16;
                    t.addr[o] = x | i << 2 | y << 5 | j << 7 | (best < 2 ? 1 << 10 : 0);
                    if (most > t.terms[o / VLX_WAVE]) t.terms[o / VLX_WAVE] = most;
                }
        }
        return t;
    }
};
template <int la, int lb, int lc, int ld>
static __device__ constexpr typename MmdDigest<la, lb, lc, ld>::Tab g_mmd_digest = MmdDigest<la, lb, lc, ld>::make();

// Orders the LDS accesses of the one wavefront of a block for the compiler; the hardware executes
// the LDS instructions of a wavefront in order.
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ double lds_at(const double* __restrict__ base, const int byte)
{
    return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(base) + byte);
}

// terms of the digestion loaded together (term counts are odd): few wavefronts a SIMD wait for LDS
// ((dd|dd) 0.336 -> 0.304 ms, (fd|dp) 1.57 -> 1.45), more of them are bound by the vector unit
// ((dp|dp) 2.49 -> 2.64); 20 waters def2-TZVP, one stream
constexpr int mmd_digest_unroll(int L) { return L >= 7 ? 5 : 1; }

// What a lane of the MD kernels keeps for the whole launch.
template <int la, int lb, int lc, int ld>
struct MmdLane {
    using S = MmdSizes<la, lb, lc, ld>;
    // byte offsets of R^0[p + q], two steps (row tile, column group) a register; masked rows and
    // columns read R^0[0] against zero rows of U
    unsigned ridx[(S::MX * S::KX + 1) / 2];
    // the lane's entries of the R recursion: byte offsets of the two sources, factor, byte offset of
    // the component of P - Q in a row of seeds
    unsigned rsrc[S::KR];
    double rfac[S::KR];
    int raxis[S::KR];
    // the lane's elements of the digestion
    int gib[S::NR], gstep[S::NR], gwrap[S::NR], gaddr[S::NR];

    __device__ __forceinline__ void init(const int lane)
    {
        static_assert(8 * S::nr < 65536 && 8 * S::nsab * S::nscd < 65536, "LDS byte offsets pack into 16 bits");
        const int lr = lane & 15, lk = lane >> 4;
#pragma unroll
        for (int e = 0; e < (S::MX * S::KX + 1) / 2; e++) ridx[e] = 0;
#pragma unroll
        for (int e = 0; e < S::MX * S::KX; e++) {
            const int p = 16 * (e / S::KX) + lr, q = 4 * (e % S::KX) + lk;
            const int tuv = g_herm.e[min(p, S::nhab - 1)] + g_herm.e[min(q, S::nhcd - 1)];
            const unsigned off = (p < S::nhab && q < S::nhcd) ? 8u * hidx_packed(tuv) : 0u;
            ridx[e / 2] |= off << (16 * (e & 1));
        }
#pragma unroll
        for (int k = 0; k < S::KR; k++) {
            const int rr = g_hrec.e[min(lane + VLX_WAVE * k, S::nr - 1)];
            rsrc[k] = 8u * (rr & 511) | 8u * ((rr >> 9) & 511) << 16;
            raxis[k] = 8 * ((rr >> 18) & 3);
            rfac[k] = static_cast<double>(rr >> 20);
        }
#pragma unroll
        for (int k = 0; k < S::NR; k++) {
            const int o = lane + VLX_WAVE * k;
            const bool ok = o < S::nout;
            gib[k] = ok ? g_mmd_digest<la, lb, lc, ld>.ib[o] : 0;
            gstep[k] = ok ? g_mmd_digest<la, lb, lc, ld>.step[o] : 0;
            gwrap[k] = ok ? g_mmd_digest<la, lb, lc, ld>.wrap[o] : 0;
            gaddr[k] = ok ? g_mmd_digest<la, lb, lc, ld>.addr[o] : 0;
        }
    }
    // element k of the digestion in D and F' (elements past the last: 0)
    __device__ __forceinline__ size_t place(const int k, const int lane, const PairInfo& bp, const PairInfo& kp,
                                            const int nao) const
    {
        const int x = gaddr[k] & 3, i = (gaddr[k] >> 2) & 7, y = (gaddr[k] >> 5) & 3, j = (gaddr[k] >> 7) & 7;
        const int row = x == 0 ? bp.ao_a + i * bp.str_a : x == 1 ? bp.ao_b + i * bp.str_b : kp.ao_a + i * kp.str_a;
        const int col = y == 1 ? bp.ao_b + j * bp.str_b : y == 2 ? kp.ao_a + j * kp.str_a : kp.ao_b + j * kp.str_b;
        return lane + VLX_WAVE * k < S::nout ? (size_t)row * nao + col : 0;
    }
    // element k's sum over its terms: integrals in outs, the six D blocks in dblk
    __device__ __forceinline__ double sum(const int k, const int terms, const double* __restrict__ outs,
                                          const double* __restrict__ dblk) const
    {
        const int step = gstep[k] & 0xffff, nv = (gstep[k] >> 16) & 0xff, wrap = gwrap[k] & 0xffff;
        int io = gib[k] & 0xffff, dof = gib[k] >> 16, c = 0;
        double v = 0.0;
        constexpr int UN = mmd_digest_unroll(S::L);
        for (int t = 0; t < terms; t += UN) {
            double x[UN], d[UN];
            // loads of several terms in flight; past the last one they repeat it
#pragma unroll
            for (int q = 0; q < UN; q++) {
                x[q] = lds_at(outs, io);
                d[q] = lds_at(dblk, dof);
                const bool more = t + q + 1 < terms, end = c + 1 == nv;
                dof += more ? 8 : 0;
                io += more ? step + (end ? wrap : 0) : 0;
                c = end ? 0 : c + 1;
            }
#pragma unroll
            for (int q = 0; q < UN; q++) v = t + q < terms ? fma(x[q], d[q], v) : v;
        }
        return v;
    }
};

// Per primitive quartet of up to 8 kets of one bra: P - Q and R^n_000 = w (-2 rho)^n F_n, n = 0..L, in
// rows of an LDS table, one lane a primitive quartet.  All of it is the same for the 64 lanes that share
// a quartet: computed there, a chain of two loads and the Boys function stood before every recursion
// (20 waters def2-TZVP, one stream: (pp|pp) 5.1 -> 4.0 ms, (fp|dp) 3.94 -> 3.78).  The rows come in the
// order in which mmd_block takes them (ket, bra primitive, ket primitive), CAP at a time.
template <int L, bool RS>
struct MmdSeeds {
    static constexpr int CAP = 16, KETS = 8, stride = (L + 4) | 1;  // odd: rows start in different banks
    static constexpr int size = CAP * stride;                      // doubles per wavefront
    const PrimPair* __restrict__ bra_prims;
    const PrimPair* __restrict__ ket_prims;
    const double* __restrict__ boys_tab;
    double omega2;
    double* rows;
    int lane, knp, kstart, before;  // lane t < KETS: primitives of ket t, first, primitive quartets before it
    int total, next, filled;        // primitive quartets of the unit, the next to be taken, in the table up to

    // kets of the unit: lane t's ket, taken or not
    __device__ __forceinline__ void open(const PairInfo& bp, const PairInfo& kp, const bool take)
    {
        knp = kp.nprim;
        kstart = kp.prim_start;
        const int n = take ? bp.nprim * knp : 0;
        int upto = n;
#pragma unroll
        for (int d = 1; d < KETS; d *= 2) {
            const int o = __shfl_up(upto, d, VLX_WAVE);
            upto += lane >= d ? o : 0;
        }
        before = upto - n;
        total = __builtin_amdgcn_readlane(upto, KETS - 1);
        next = filled = 0;
    }
    // row of the next primitive quartet
    __device__ __forceinline__ const double* take(const PairInfo& bp)
    {
        if (next == filled) fill(bp);
        return rows + (next++ - (filled - CAP)) * stride;
    }
    __device__ __forceinline__ void fill(const PairInfo& bp)
    {
        wave_lds_fence();
        const int c = min(filled + lane, total - 1);
        int t = 0;
#pragma unroll
        for (int k = 1; k < KETS; k++) t = c >= __builtin_amdgcn_readlane(before, k) ? k : t;
        const int r = c - __shfl(before, t, VLX_WAVE), nk = __shfl(knp, t, VLX_WAVE), k0 = __shfl(kstart, t, VLX_WAVE);
        const int ib = static_cast<int>((static_cast<float>(r) + 0.5f) / static_cast<float>(nk)), ik = r - ib * nk;
        const PrimPair pb = bra_prims[bp.prim_start + ib];
        const PrimPair pk = ket_prims[k0 + ik];
        const double sz = pb.zeta + pk.zeta;
        const double rho_c = pb.zeta * pk.zeta * vrcp<double>(sz);
        double rho = rho_c, w = vrsqrt<double>(sz);
        if constexpr (RS) {
            const double sfac = omega2 / (omega2 + rho_c);
            rho = rho_c * sfac;
            w *= sqrt(sfac);
        }
        const double pqx = pb.px - pk.px, pqy = pb.py - pk.py, pqz = pb.pz - pk.pz;
        double seed[L + 1];
        boys_eval<L, double, true>(rho * (pqx * pqx + pqy * pqy + pqz * pqz), boys_tab, seed);
        if (lane < CAP) {
            double* row = rows + lane * stride;
            row[0] = pqx;
            row[1] = pqy;
            row[2] = pqz;
#pragma unroll
            for (int n = 0; n <= L; n++) {
                row[3 + n] = w * seed[n];
                w *= -2.0 * rho;
            }
        }
        filled += CAP;
        wave_lds_fence();
    }
};

// Contracted spherical block (ab|cd) of one shell quartet by one wavefront, into outs[ab][cd] (LDS).
// rbuf: R^n for even n in the first nr doubles, odd n in the second.
template <int la, int lb, int lc, int ld, bool RS>
__device__ __forceinline__ void mmd_block(const MmdLane<la, lb, lc, ld>& ln, const int lane, const PairInfo& bp,
                                          const PairInfo& kp, const double* __restrict__ bra_u,
                                          const double* __restrict__ ket_u, MmdSeeds<la + lb + lc + ld, RS>& seeds,
                                          double* __restrict__ rbuf, double* __restrict__ outs)
{
    using S = MmdSizes<la, lb, lc, ld>;
    constexpr int L = S::L, MX = S::MX, KX = S::KX, MT = S::MT, NT = S::NT, KR = S::KR;
    const int lr = lane & 15, lk = lane >> 4;
    vlx_d4 acc[NT][MT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int m = 0; m < MT; m++) acc[nt][m] = vlx_d4{0.0, 0.0, 0.0, 0.0};
    for (int ib = 0; ib < bp.nprim; ib++) {
        const double* ua = bra_u + (size_t)(bp.prim_start + ib) * (S::HA * S::SA) + lk * S::SA + lr;
        vlx_d4 x[S::XSUM ? NT : 1][MX];
        auto clear_x = [&](vlx_d4 (&t)[MX]) {
#pragma unroll
            for (int m = 0; m < MX; m++) t[m] = vlx_d4{0.0, 0.0, 0.0, 0.0};
        };
        // out[ab][cd] += sum_p U_AB[p][ab] X[p][cd] of column tile nt
        auto out_product = [&](const vlx_d4 (&t)[MX], vlx_d4 (&o)[MT]) {
#pragma unroll
            for (int kp2 = 0; kp2 < S::KO; kp2++) {
#pragma unroll
                for (int ms = 0; ms < MT; ms++)
                    o[ms] = __builtin_amdgcn_mfma_f64_16x16x4f64(ua[4 * kp2 * S::SA + 16 * ms], t[kp2 / 4][kp2 % 4],
                                                                o[ms], 0, 0, 0);
            }
        };
        if constexpr (S::XSUM) {
#pragma unroll
            for (int nt = 0; nt < NT; nt++) clear_x(x[nt]);
        }
        for (int ik = 0; ik < kp.nprim; ik++) {
            const double* uc = ket_u + (size_t)(kp.prim_start + ik) * (S::HC * S::SC) + lk * S::SC + lr;
            double ucv[S::PRE_X ? NT : 1][S::PRE_X ? KX : 1];
            if constexpr (S::PRE_X) {
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
#pragma unroll
                    for (int kq = 0; kq < KX; kq++) ucv[nt][kq] = uc[4 * kq * S::SC + 16 * nt];
            }
            const double* row = seeds.take(bp);
            double pq[KR], seed[L + 1];
#pragma unroll
            for (int k = 0; k < KR; k++) pq[k] = lds_at(row, ln.raxis[k]);
#pragma unroll
            for (int n = 0; n <= L; n++) seed[n] = row[3 + n];
            // R levels n = L .. 0, one FMA and one product per entry
            if (lane == 0) rbuf[(L & 1) * S::nr] = seed[L];
#pragma unroll
            for (int n = L - 1; n >= 0; n--) {
                wave_lds_fence();
                const double* prev = rbuf + ((n + 1) & 1) * S::nr;
                double* cur = rbuf + (n & 1) * S::nr;
#pragma unroll
                for (int k = 0; VLX_WAVE * k < nherm(L - n); k++) {
                    const int idx = lane + VLX_WAVE * k;
                    if (idx < nherm(L - n)) {
                        const double v1 = lds_at(prev, ln.rsrc[k] & 0xffff), v2 = lds_at(prev, ln.rsrc[k] >> 16);
                        const double val = fma(ln.rfac[k], v2, pq[k] * v1);
                        cur[idx] = idx == 0 ? seed[n] : val;
                    }
                }
            }
            wave_lds_fence();
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                vlx_d4 (&t)[MX] = x[S::XSUM ? nt : 0];
                if constexpr (!S::XSUM) clear_x(t);
#pragma unroll
                for (int kq = 0; kq < KX; kq++) {
                    double bv;
                    if constexpr (S::PRE_X) bv = ucv[nt][kq];
                    else bv = uc[4 * kq * S::SC + 16 * nt];
#pragma unroll
                    for (int m = 0; m < MX; m++) {
                        const int e = m * KX + kq;
                        const double av = lds_at(rbuf, (e & 1) ? ln.ridx[e / 2] >> 16 : ln.ridx[e / 2] & 0xffff);
                        t[m] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, t[m], 0, 0, 0);
                    }
                }
                if constexpr (!S::XSUM) out_product(t, acc[nt]);
            }
            wave_lds_fence();
        }
        if constexpr (S::XSUM) {
#pragma unroll
            for (int nt = 0; nt < NT; nt++) out_product(x[nt], acc[nt]);
        }
    }
    // contracted block -> LDS [ab][cd]
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int ms = 0; ms < MT; ms++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int ab = 16 * ms + lk + 4 * r, cd = 16 * nt + lr;
                if (ab < S::nsab && cd < S::nscd) outs[ab * S::nscd + cd] = acc[nt][ms][r];
            }
}

// Direct digestion (several densities, deterministic builds, tiles that do not fit in LDS): work item
// {j0, i0, i1}, bra i0 with kets [j0, i1), one shell quartet at a time, F' through global atomics.
// With a.ndens > 1 each block is digested into every density (density d at D0 + d * dstride, its F' at
// F0 + d * dstride, factors dfac[2 d], dfac[2 d + 1]).  a.det: F0 holds fixed-point accumulators
// (fx_add, two words per element) and the factors come from dfac also for one density.
template <int la, int lb, int lc, int ld, bool RS>
__global__ void __launch_bounds__(VLX_WAVE) __attribute__((amdgpu_waves_per_eu(MmdSizes<la, lb, lc, ld>::occupancy)))
    fock_kernel_mmd(const PairInfo* __restrict__ bra, const PrimPair* __restrict__ bra_prims,
                    const double* __restrict__ bra_u, const PairInfo* __restrict__ ket,
                    const PrimPair* __restrict__ ket_prims, const double* __restrict__ ket_u,
                    const WorkItem* __restrict__ items, const double* __restrict__ boys_tab,
                    const double* __restrict__ D0, double* __restrict__ F0, const MolDesc* __restrict__ mols,
                    const int* __restrict__ glim, const double* __restrict__ dfac, const FockScalars a)
{
    using S = MmdSizes<la, lb, lc, ld>;
    constexpr int NR = S::NR;
    __shared__ double rbuf[2 * S::nr];
    __shared__ double outs[S::nsab * S::nscd];
    __shared__ double dblk[S::nout];
    __shared__ double rows[MmdSeeds<S::L, RS>::size];
    const int lane = threadIdx.x;
    MmdLane<la, lb, lc, ld> ln;
    ln.init(lane);
    MmdSeeds<S::L, RS> seeds{bra_prims, ket_prims, boys_tab, a.omega2, rows, lane};
    unsigned long long taken = 0;
    for (long long it = blockIdx.x; it < a.nitems; it += gridDim.x) {
        const WorkItem wi = items[it];
        const MolDesc md = mols[wi.mol];
        const PairInfo bp = bra[wi.i0];
        for (int j = wi.j0; j < wi.i1; j++) {
            // kets in units of up to 8; density-weighted screening (one quartet per wavefront)
            if (((j - wi.j0) % MmdSeeds<S::L, RS>::KETS) == 0) {
                const int n = min(wi.i1 - j, MmdSeeds<S::L, RS>::KETS);
                const PairInfo kl = ket[j + min(lane, n - 1)];
                const bool take = lane < n && (glim == nullptr || bp.bin + kl.bin <= quartet_bin_limit(glim, a.ngroups, bp.grp_a, bp.grp_b, kl.grp_a, kl.grp_b));
                taken = __ballot(take);
                seeds.open(bp, kl, take);
            }
            const int t = (j - wi.j0) % MmdSeeds<S::L, RS>::KETS;
            if (!((taken >> t) & 1)) continue;
            const PairInfo kp = ket[j];
            // elements of the six blocks: their place in D and F', and the first density's D
            size_t goff[NR];
            double dval[NR];
#pragma unroll
            for (int k = 0; k < NR; k++) {
                goff[k] = ln.place(k, lane, bp, kp, md.nao);
                dval[k] = D0[md.base + goff[k]];
            }
            mmd_block<la, lb, lc, ld, RS>(ln, lane, bp, kp, bra_u, ket_u, seeds, rbuf, outs);
            double sf = 1.0;
            if (bp.same) sf *= 0.5;
            if (kp.same) sf *= 0.5;
            if (a.same_class && bp.rank == j) sf *= 0.5;
            const int nds = a.ndens > 1 ? a.ndens : 1;
            for (int dd = 0; dd < nds; dd++) {
                if (dd > 0) {
                    wave_lds_fence();
#pragma unroll
                    for (int k = 0; k < NR; k++) dval[k] = D0[md.base + dd * a.dstride + goff[k]];
                }
#pragma unroll
                for (int k = 0; k < NR; k++)
                    if (lane + VLX_WAVE * k < S::nout) dblk[ln.gwrap[k] >> 16] = dval[k];
                wave_lds_fence();
                const bool table = a.det || a.ndens > 1;
                const double fj = sf * (table ? dfac[2 * dd] : a.fj), fk = sf * (table ? dfac[2 * dd + 1] : a.fk);
#pragma unroll
                for (int k = 0; k < NR; k++) {
                    const double coef = (ln.gaddr[k] >> 10) & 1 ? fj : fk;
                    const int terms = coef != 0.0 ? ln.gstep[k] >> 24 : 0;
                    const double v = ln.sum(k, terms, outs, dblk);
                    if (terms > 0) {
                        const size_t at = md.base + dd * a.dstride + goff[k];
                        if (a.det) fx_add(reinterpret_cast<unsigned long long*>(F0), at, coef * v);
                        else unsafeAtomicAdd(F0 + at, coef * v);
                    }
                }
            }
            wave_lds_fence();
        }
    }
}

// Tiled digestion: a block of NW wavefronts takes one TileItem (here [j0, j1) are ket pairs of the
// tiled order), and the F' elements go into the six LDS tiles of the item's atom groups, flushed once
// per item as in fock_kernel_tiled.  The direct form is bound by its global atomics: FP64 atomics of
// eight L2s are carried out at the memory side, 13 to 17 billion a second over the whole chip in every
// class, while the matrix cores are busy 17% and the vector units 26% of the time ((fp|dp), 116 atomics
// a quartet).  Units of up to 8 kets of one bra go round the wavefronts.  One stream, 20 waters
// def2-TZVP, direct / tiled: (fp|dp) 4.3 / 3.9 ms, (fp|fp) 1.5 / 1.8 ms (its tiles leave 8 wavefronts a
// CU), (dd|dp) of one water 0.043 / 0.043 ms.
template <int la, int lb, int lc, int ld>
struct MmdTile {
    using S = MmdSizes<la, lb, lc, ld>;
    static constexpr int NW = 4 * S::occupancy;  // one block fills a CU's registers
    static constexpr int scratch = 2 * S::nr + S::nsab * S::nscd + S::nout + MmdSeeds<S::L, false>::size;  // doubles per wavefront
    static constexpr int KETS = MmdSeeds<S::L, false>::KETS;
};

template <int la, int lb, int lc, int ld, bool RS>
__global__ void __launch_bounds__((MmdTile<la, lb, lc, ld>::NW * VLX_WAVE))
    __attribute__((amdgpu_waves_per_eu(MmdSizes<la, lb, lc, ld>::occupancy)))
    fock_kernel_mmd_tiled(const PairInfo* __restrict__ pairs_bra, const PrimPair* __restrict__ bra_prims,
                          const double* __restrict__ bra_u, const PairInfo* __restrict__ pairs_ket,
                          const PrimPair* __restrict__ ket_prims, const double* __restrict__ ket_u,
                          const TileItem* __restrict__ items, const double* __restrict__ boys_tab,
                          const double* __restrict__ D0, double* __restrict__ F0, const MolDesc* __restrict__ mols,
                          const int* __restrict__ glim, const int* __restrict__ grp_off, const int* __restrict__ grp_n,
                          const int* __restrict__ grp_ao, const FockScalars a)
{
    using S = MmdSizes<la, lb, lc, ld>;
    using T = MmdTile<la, lb, lc, ld>;
    constexpr int NR = S::NR, NW = T::NW;
    extern __shared__ double tiles[];
    const int lane = threadIdx.x & (VLX_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / VLX_WAVE);
    double* rbuf = tiles + a.tile_doubles + wave * T::scratch;
    double* outs = rbuf + 2 * S::nr;
    double* dblk = outs + S::nsab * S::nscd;
    MmdSeeds<S::L, RS> seeds{bra_prims, ket_prims, boys_tab, a.omega2, dblk + S::nout, lane};
    for (int e = threadIdx.x; e < a.tile_doubles; e += NW * VLX_WAVE) tiles[e] = 0.0;
    MmdLane<la, lb, lc, ld> ln;
    ln.init(lane);
    __syncthreads();
    for (long long it = blockIdx.x; it < a.nitems; it += gridDim.x) {
        const TileItem ti = items[it];
        const MolDesc md = mols[ti.mol];
        const double* __restrict__ D = D0 + md.base;
        double* __restrict__ F = F0 + md.base;
        int ilim = a.ithreshold;
        if (glim != nullptr) ilim = min(ilim, quartet_bin_limit(glim, a.ngroups, ti.ga, ti.gb, ti.gc, ti.gd));
        // smallest bin sum of the item: past the limit it has no quartet (block-uniform skip)
        if (a.ithreshold >= 0 && pairs_bra[ti.i0].bin + ti.bin_lo > ilim) continue;
        const int nA = grp_n[ti.ga * 4 + la], nB = grp_n[ti.gb * 4 + lb];
        const int nC = grp_n[ti.gc * 4 + lc], nD = grp_n[ti.gd * 4 + ld];
        // tiles J_AB, K_AC, K_BC, J_CD, K_AD, K_BD
        double* t_jab = tiles;
        double* t_kac = t_jab + nA * nB;
        double* t_kbc = t_kac + nA * nC;
        double* t_jcd = t_kbc + nB * nC;
        double* t_kad = t_jcd + nC * nD;
        double* t_kbd = t_kad + nA * nD;
        // the lane's elements in the tiles: place of component (i, j), row stride
        int tbase[NR], tstride[NR];
#pragma unroll
        for (int k = 0; k < NR; k++) {
            const int x = ln.gaddr[k] & 3, i = (ln.gaddr[k] >> 2) & 7, y = (ln.gaddr[k] >> 5) & 3, j = (ln.gaddr[k] >> 7) & 7;
            tstride[k] = y == 1 ? nB : y == 2 ? nC : nD;
            const double* t = y == 1 ? t_jab : y == 2 ? (x == 0 ? t_kac : t_kbc) : x == 0 ? t_kad : x == 1 ? t_kbd : t_jcd;
            tbase[k] = static_cast<int>(t - tiles) + i * tstride[k] + j;
        }
        // kets of a unit: fewer where the item has few, for about 8 units a wavefront (8 kets always left
        // wavefronts idle at the end of items: (dd|dd) 0.30 -> 0.18 ms, (fp|dp) 3.8 -> 3.35 ms, (fp|dp) of
        // two waters 0.17 -> 0.10 ms)
        const int ku = max(1, min(T::KETS, (ti.i1 - ti.i0) * (ti.j1 - ti.j0) / (8 * NW)));
        const int nunit = (ti.j1 - ti.j0 + ku - 1) / ku;
        for (int u = wave; u < (ti.i1 - ti.i0) * nunit; u += NW) {
            const int i = ti.i0 + u / nunit, j0 = ti.j0 + u % nunit * ku;
            const PairInfo bp = pairs_bra[i];
            const int n = min(ti.j1 - j0, ku);
            const PairInfo kl = pairs_ket[j0 + min(lane, n - 1)];
            const bool take = lane < n && !(a.ithreshold >= 0 && bp.bin + kl.bin > ilim) &&
                              !(a.same_class && bp.rank < kl.rank);
            const unsigned long long taken = __ballot(take);
            if (taken == 0) continue;
            seeds.open(bp, kl, take);
            for (int t = 0; t < n; t++) {
                if (!((taken >> t) & 1)) continue;
                const PairInfo kp = pairs_ket[j0 + t];
                int toff[NR];
                double dval[NR];
#pragma unroll
                for (int k = 0; k < NR; k++) {
                    const int x = ln.gaddr[k] & 3, y = (ln.gaddr[k] >> 5) & 3;
                    const int row = x == 0 ? bp.loc_a : x == 1 ? bp.loc_b : kp.loc_a;
                    const int col = y == 1 ? bp.loc_b : y == 2 ? kp.loc_a : kp.loc_b;
                    toff[k] = tbase[k] + row * tstride[k] + col;
                    dval[k] = D[ln.place(k, lane, bp, kp, md.nao)];
                }
                mmd_block<la, lb, lc, ld, RS>(ln, lane, bp, kp, bra_u, ket_u, seeds, rbuf, outs);
                double sf = 1.0;
                if (bp.same) sf *= 0.5;
                if (kp.same) sf *= 0.5;
                if (a.same_class && bp.rank == kp.rank) sf *= 0.5;
#pragma unroll
                for (int k = 0; k < NR; k++)
                    if (lane + VLX_WAVE * k < S::nout) dblk[ln.gwrap[k] >> 16] = dval[k];
                wave_lds_fence();
#pragma unroll
                for (int k = 0; k < NR; k++) {
                    const int terms = ((ln.gaddr[k] >> 10) & 1 ? a.fj : a.fk) != 0.0 ? ln.gstep[k] >> 24 : 0;
                    const double v = ln.sum(k, terms, outs, dblk);
                    if (terms > 0) unsafeAtomicAdd(&tiles[toff[k]], sf * v);
                }
                wave_lds_fence();
            }
        }
        __syncthreads();
        const int* ra = grp_ao + grp_off[ti.ga * 4 + la];
        const int* rb = grp_ao + grp_off[ti.gb * 4 + lb];
        const int* rc = grp_ao + grp_off[ti.gc * 4 + lc];
        const int* rd = grp_ao + grp_off[ti.gd * 4 + ld];
        if (a.fj != 0.0) {
            flush_tile<NW>(F, md.nao, t_jab, nA, nB, ra, rb, a.fj, wave, lane);
            flush_tile<NW>(F, md.nao, t_jcd, nC, nD, rc, rd, a.fj, wave, lane);
        }
        if (a.fk != 0.0) {
            flush_tile<NW>(F, md.nao, t_kac, nA, nC, ra, rc, a.fk, wave, lane);
            flush_tile<NW>(F, md.nao, t_kbc, nB, nC, rb, rc, a.fk, wave, lane);
            flush_tile<NW>(F, md.nao, t_kad, nA, nD, ra, rd, a.fk, wave, lane);
            flush_tile<NW>(F, md.nao, t_kbd, nB, nD, rb, rd, a.fk, wave, lane);
        }
        __syncthreads();
    }
}

template <int la, int lb, int lc, int ld>
__global__ void __launch_bounds__(VLX_WAVE) eri_out_kernel_md(const EriArgs a)
{
    using S = md::Sizes<la, lb, lc, ld>;
    __shared__ double tab_lds[S::tab_in_lds ? BOYS_TAB_SIZE : 1];
    __shared__ double work[S::lds];
    __shared__ double out[S::nsab * S::nscd];
    const double* tab = S::tab_in_lds ? tab_lds : a.boys_tab;
    if constexpr (S::tab_in_lds) stage_boys<true>(tab_lds, a.boys_tab);
    for (int qi = blockIdx.x; qi < a.nquartets; qi += gridDim.x) {
        const int2 qq = a.quartets[qi];
        const PairInfo bp = a.bra[qq.x];
        const PairInfo kp = a.ket[qq.y];
        const double abv[3] = {bp.abx, bp.aby, bp.abz}, cdv[3] = {kp.abx, kp.aby, kp.abz};
        md::quartet<la, lb, lc, ld>(a.bra_prims + bp.prim_start, bp.nprim, abv, a.ket_prims + kp.prim_start,
                                    kp.nprim, cdv, tab, 0.0, work, out);
        for (int k = threadIdx.x; k < S::nsab * S::nscd; k += blockDim.x)
            a.out[(size_t)qi * S::nsab * S::nscd + k] = out[k];
        __syncthreads();
    }
}

template <int la, int lb>
__global__ void __launch_bounds__(VLX_WAVE) diag_kernel_md(const DiagArgs a)
{
    using S = md::Sizes<la, lb, la, lb>;
    __shared__ double tab_lds[S::tab_in_lds ? BOYS_TAB_SIZE : 1];
    __shared__ double work[S::lds];
    __shared__ double out[S::nsab * S::nscd];
    const double* tab = S::tab_in_lds ? tab_lds : a.boys_tab;
    if constexpr (S::tab_in_lds) stage_boys<true>(tab_lds, a.boys_tab);
    for (int pi = blockIdx.x; pi < a.npairs; pi += gridDim.x) {
        const PairInfo pp = a.pairs[pi];
        const double abv[3] = {pp.abx, pp.aby, pp.abz};
        md::quartet<la, lb, la, lb>(a.prims + pp.prim_start, pp.nprim, abv, a.prims + pp.prim_start, pp.nprim, abv,
                                    tab, 0.0, work, out);
        double mx = 0.0;
        for (int k = threadIdx.x; k < S::nsab * S::nscd; k += blockDim.x) mx = (mx < out[k]) ? out[k] : mx;
        for (int off = 32; off > 0; off >>= 1) {
            const double o = __shfl_xor(mx, off, VLX_WAVE);
            mx = (mx < o) ? o : mx;
        }
        if (threadIdx.x == 0) a.maxval[pi] = mx;
        __syncthreads();
    }
}

// Fock: the matrix-core kernel (U arrays of both pair sets in FockArgs); the
// cooperative LDS kernel serves explicit quartets and the screener.
#define VLX_MMD_LAUNCH(la, lb, lc, ld, RS)                                                              \
    hipLaunchKernelGGL((fock_kernel_mmd<la, lb, lc, ld, RS>), dim3(g), dim3(VLX_WAVE), 0, s, a.bra,     \
                       a.bra_prims, a.bra_u, a.ket, a.ket_prims, a.ket_u, a.items, a.boys_tab, a.D, a.F, \
                       a.mols, a.glim, a.dfac, a.sc)
// tiled digestion: TileItem list, dynamic LDS of the tiles (a.tile_lds_bytes) and the waves' scratch
#define VLX_INSTANTIATE_MMD_TILED(la, lb, lc, ld)                                                       \
    void launch_mmd_tiled_##la##lb##lc##ld(const FockArgs& a, int grid, hipStream_t s)                  \
    {                                                                                                   \
        using T = MmdTile<la, lb, lc, ld>;                                                              \
        const int lds = a.tile_lds_bytes + 8 * T::NW * T::scratch;                                      \
        if (a.sc.omega2 > 0.0)                                                                          \
            hipLaunchKernelGGL((fock_kernel_mmd_tiled<la, lb, lc, ld, true>), dim3(grid), dim3(T::NW * VLX_WAVE), \
                               lds, s, a.bra, a.bra_prims, a.bra_u, a.ket, a.ket_prims, a.ket_u, a.titems, \
                               a.boys_tab, a.D, a.F, a.mols, a.glim, a.grp_off, a.grp_n, a.grp_ao, a.sc); \
        else                                                                                            \
            hipLaunchKernelGGL((fock_kernel_mmd_tiled<la, lb, lc, ld, false>), dim3(grid),              \
                               dim3(T::NW * VLX_WAVE), lds, s, a.bra, a.bra_prims, a.bra_u, a.ket,      \
                               a.ket_prims, a.ket_u, a.titems, a.boys_tab, a.D, a.F, a.mols, a.glim,    \
                               a.grp_off, a.grp_n, a.grp_ao, a.sc);                                     \
    }                                                                                                   \
    int mmd_scratch_##la##lb##lc##ld() { return 8 * MmdTile<la, lb, lc, ld>::NW * MmdTile<la, lb, lc, ld>::scratch; }
// launch_mmd_: the matrix-core kernel as an alternative variant of a class
// whose default kernel is generated (same MD work items).
#define VLX_INSTANTIATE_MMD(la, lb, lc, ld)                                                             \
    void launch_mmd_##la##lb##lc##ld(const FockArgs& a, int grid, hipStream_t s)                        \
    {                                                                                                   \
        const int g = grid > 0 ? grid : static_cast<int>(std::min<long long>(a.sc.nitems, 16384));       \
        if (a.sc.omega2 > 0.0) VLX_MMD_LAUNCH(la, lb, lc, ld, true);                                    \
        else VLX_MMD_LAUNCH(la, lb, lc, ld, false);                                                     \
    }
#define VLX_INSTANTIATE_MD_CLASS(la, lb, lc, ld)                                                        \
    void launch_fock_##la##lb##lc##ld(const FockArgs& a, int grid, hipStream_t s)                       \
    {                                                                                                   \
        const int g = grid > 0 ? grid : static_cast<int>(std::min<long long>(a.sc.nitems, 16384));       \
        if (a.sc.omega2 > 0.0) VLX_MMD_LAUNCH(la, lb, lc, ld, true);                                    \
        else VLX_MMD_LAUNCH(la, lb, lc, ld, false);                                                     \
    }                                                                                                   \
    void launch_eri_##la##lb##lc##ld(const EriArgs& a, hipStream_t s)                                   \
    {                                                                                                   \
        const int g = std::min(a.nquartets, 4096);                                                      \
        hipLaunchKernelGGL((eri_out_kernel_md<la, lb, lc, ld>), dim3(g), dim3(VLX_WAVE), 0, s, a);      \
    }

#define VLX_INSTANTIATE_MD_DIAG(la, lb)                                                                 \
    void launch_diag_##la##lb(const DiagArgs& a, hipStream_t s)                                         \
    {                                                                                                   \
        const int g = std::min(a.npairs, 4096);                                                         \
        hipLaunchKernelGGL((diag_kernel_md<la, lb>), dim3(g), dim3(VLX_WAVE), 0, s, a);                 \
    }
