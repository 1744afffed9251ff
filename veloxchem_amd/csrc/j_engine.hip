// Hermite densities of the Coulomb build, its kernels for every pair of Hermite ranks, and the
// transformation of J_p to F' (j_kernels.h).
#include <algorithm>

#include "j_kernels.h"
#include "md_kernels.h"

namespace {

// One primitive pair's E^{ij}_t per axis, i <= la, j <= lb, without the prefactor.
template <int la, int lb>
__device__ __forceinline__ void j_expand(const PrimPair& pr, const PairInfo& pp, double (&E)[3][la + 1][lb + 1][la + lb + 1])
{
    const double h = 0.5 / pr.zeta;
    const double pa[3] = {pr.pax, pr.pay, pr.paz};
    const double pb[3] = {pr.pax + pp.abx, pr.pay + pp.aby, pr.paz + pp.abz};
#pragma unroll
    for (int x = 0; x < 3; x++) {
#pragma unroll
        for (int i = 0; i <= la; i++)
#pragma unroll
            for (int j = 0; j <= lb; j++)
#pragma unroll
                for (int t = 0; t <= la + lb; t++) {
                    if (i == 0 && j == 0) {
                        E[x][0][0][t] = t == 0 ? 1.0 : 0.0;
                        continue;
                    }
                    if (t > i + j) {
                        E[x][i][j][t] = 0.0;
                        continue;
                    }
                    // raise i along j = 0, then j
                    const double (&f)[la + lb + 1] = j > 0 ? E[x][i][j - 1] : E[x][i - 1][j];
                    const double d = j > 0 ? pb[x] : pa[x];
                    double s = d * f[t];
                    if (t > 0) s = fma(h, f[t - 1], s);
                    if (t + 1 <= la + lb) s = fma(t + 1.0, f[t + 1], s);
                    E[x][i][j][t] = s;
                }
    }
}

constexpr int j_cart(int l, int idx, int axis)  // exponent of Cartesian function idx: x falling, then y
{
    int k = 0;
    for (int x = l; x >= 0; x--)
        for (int y = l - x; y >= 0; y--, k++)
            if (k == idx) return axis == 0 ? x : axis == 1 ? y : l - x - y;
    return 0;
}

// visit(s, h, c): U[h][s] gains c, for every term of the Hermite-to-spherical matrix of one primitive
template <int la, int lb, class F>
__device__ __forceinline__ void j_terms(const double (&E)[3][la + 1][lb + 1][la + lb + 1], F&& visit)
{
#pragma unroll
    for (int a = 0; a < 2 * la + 1; a++) {
        int cia[3] = {0, 0, 0};
        double cfa[3] = {0.0, 0.0, 0.0};
        const int nta = md::sph_terms(la, a, cia, cfa);
#pragma unroll
        for (int b = 0; b < 2 * lb + 1; b++) {
            int cib[3] = {0, 0, 0};
            double cfb[3] = {0.0, 0.0, 0.0};
            const int ntb = md::sph_terms(lb, b, cib, cfb);
#pragma unroll
            for (int ia = 0; ia < 3; ia++)
#pragma unroll
                for (int ib = 0; ib < 3; ib++) {
                    if (ia >= nta || ib >= ntb) continue;
                    const int ax = j_cart(la, cia[ia], 0), ay = j_cart(la, cia[ia], 1), az = j_cart(la, cia[ia], 2);
                    const int bx = j_cart(lb, cib[ib], 0), by = j_cart(lb, cib[ib], 1), bz = j_cart(lb, cib[ib], 2);
                    const double c = cfa[ia] * cfb[ib];
                    for (int t = 0; t <= ax + bx; t++)
                        for (int u = 0; u <= ay + by; u++)
                            for (int v = 0; v <= az + bz; v++)
                                visit(a * (2 * lb + 1) + b, j_index(t, u, v),
                                      c * E[0][ax][bx][t] * E[1][ay][by][u] * E[2][az][bz][v], (t + u + v) & 1);
                }
        }
    }
}

// Row of the entry of each primitive of a pair class: zeta, P and H; its J_p cleared.
template <int la, int lb>
__global__ void __launch_bounds__(256)
    j_density_kernel(const PairInfo* __restrict__ pairs, const PrimPair* __restrict__ prims,
                     const int* __restrict__ pair_of, const int* __restrict__ entry0, int nprims,
                     const double* __restrict__ D, int nao, double* __restrict__ rows, double* __restrict__ jp)
{
    constexpr int NH = j_nherm(la + lb), NS = (2 * la + 1) * (2 * lb + 1);
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= nprims) return;
    const int pi = pair_of[p];
    const PairInfo pp = pairs[pi];
    const PrimPair pr = prims[p];
    const int e = entry0[pi] + p - pp.prim_start;
    double E[3][la + 1][lb + 1][la + lb + 1];
    j_expand<la, lb>(pr, pp, E);
    double d[NS], H[NH];
    const double k = pp.same ? 0.5 * pr.k : pr.k;
    for (int a = 0; a < 2 * la + 1; a++)
        for (int b = 0; b < 2 * lb + 1; b++)
            d[a * (2 * lb + 1) + b] = k * D[(size_t)(pp.ao_a + a * pp.str_a) * nao + pp.ao_b + b * pp.str_b];
    for (int h = 0; h < NH; h++) H[h] = 0.0;
    j_terms<la, lb>(E, [&](int s, int h, double c, int odd) { H[h] = fma(odd ? -c : c, d[s], H[h]); });
    double* row = rows + (size_t)e * j_row(la + lb);
    row[0] = pr.zeta;
    row[1] = pr.px;
    row[2] = pr.py;
    row[3] = pr.pz;
    for (int h = 0; h < NH; h++) {
        row[4 + h] = H[h];
        jp[(size_t)e * NH + h] = 0.0;
    }
}

// F'_ab += factor sum_p U_ab[p] J_p of each primitive of a pair class.
template <int la, int lb>
__global__ void __launch_bounds__(256)
    j_fock_kernel(const PairInfo* __restrict__ pairs, const PrimPair* __restrict__ prims,
                  const int* __restrict__ pair_of, const int* __restrict__ entry0, int nprims,
                  const double* __restrict__ jp, double factor, int nao, double* __restrict__ F)
{
    constexpr int NH = j_nherm(la + lb), NS = (2 * la + 1) * (2 * lb + 1);
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= nprims) return;
    const int pi = pair_of[p];
    const PairInfo pp = pairs[pi];
    const PrimPair pr = prims[p];
    const int e = entry0[pi] + p - pp.prim_start;
    double E[3][la + 1][lb + 1][la + lb + 1];
    j_expand<la, lb>(pr, pp, E);
    double out[NS], J[NH];
    for (int h = 0; h < NH; h++) J[h] = jp[(size_t)e * NH + h];
    for (int s = 0; s < NS; s++) out[s] = 0.0;
    j_terms<la, lb>(E, [&](int s, int h, double c, int) { out[s] = fma(c, J[h], out[s]); });
    const double k = factor * (pp.same ? 0.5 * pr.k : pr.k);
    for (int a = 0; a < 2 * la + 1; a++)
        for (int b = 0; b < 2 * lb + 1; b++)
            unsafeAtomicAdd(F + (size_t)(pp.ao_a + a * pp.str_a) * nao + pp.ao_b + b * pp.str_b,
                            k * out[a * (2 * lb + 1) + b]);
}

template <int la, int lb>
void density(const JPrep& a, hipStream_t s)
{
    hipLaunchKernelGGL((j_density_kernel<la, lb>), dim3((a.nprims + 255) / 256), dim3(256), 0, s, a.pairs, a.prims,
                       a.pair_of, a.entry0, a.nprims, a.D, a.nao, a.rows, a.jp);
}
template <int la, int lb>
void fock(const JPrep& a, hipStream_t s)
{
    hipLaunchKernelGGL((j_fock_kernel<la, lb>), dim3((a.nprims + 255) / 256), dim3(256), 0, s, a.pairs, a.prims,
                       a.pair_of, a.entry0, a.nprims, a.jp, a.factor, a.nao, a.F);
}

template <int LAB, int LCD>
void coulomb(const JArgs& a, hipStream_t s)
{
    const int g = std::min(a.nitems, 65536);
    if (a.omega2 > 0.0) hipLaunchKernelGGL((j_kernel<LAB, LCD, true>), dim3(g), dim3(JBLOCK), 0, s, a);
    else hipLaunchKernelGGL((j_kernel<LAB, LCD, false>), dim3(g), dim3(JBLOCK), 0, s, a);
}

}  // namespace

void vlx_launch_j_density(int la, int lb, const JPrep& a, hipStream_t s)
{
    if (a.nprims <= 0) return;
    switch (4 * la + lb) {
    case 0: return density<0, 0>(a, s);
    case 4: return density<1, 0>(a, s);
    case 5: return density<1, 1>(a, s);
    case 8: return density<2, 0>(a, s);
    case 9: return density<2, 1>(a, s);
    case 10: return density<2, 2>(a, s);
    case 12: return density<3, 0>(a, s);
    case 13: return density<3, 1>(a, s);
    case 14: return density<3, 2>(a, s);
    case 15: return density<3, 3>(a, s);
    }
}

void vlx_launch_j_fock(int la, int lb, const JPrep& a, hipStream_t s)
{
    if (a.nprims <= 0) return;
    switch (4 * la + lb) {
    case 0: return fock<0, 0>(a, s);
    case 4: return fock<1, 0>(a, s);
    case 5: return fock<1, 1>(a, s);
    case 8: return fock<2, 0>(a, s);
    case 9: return fock<2, 1>(a, s);
    case 10: return fock<2, 2>(a, s);
    case 12: return fock<3, 0>(a, s);
    case 13: return fock<3, 1>(a, s);
    case 14: return fock<3, 2>(a, s);
    case 15: return fock<3, 3>(a, s);
    }
}

void vlx_launch_j(int lab, int lcd, const JArgs& a, hipStream_t s)
{
    if (a.nitems <= 0) return;
    switch (8 * lab + lcd) {
#define VLX_J(LAB, LCD) \
    case 8 * LAB + LCD: return coulomb<LAB, LCD>(a, s);
        VLX_J(0, 0) VLX_J(0, 1) VLX_J(0, 2) VLX_J(0, 3) VLX_J(0, 4) VLX_J(0, 5) VLX_J(0, 6)
        VLX_J(1, 0) VLX_J(1, 1) VLX_J(1, 2) VLX_J(1, 3) VLX_J(1, 4) VLX_J(1, 5) VLX_J(1, 6)
        VLX_J(2, 0) VLX_J(2, 1) VLX_J(2, 2) VLX_J(2, 3) VLX_J(2, 4) VLX_J(2, 5) VLX_J(2, 6)
        VLX_J(3, 0) VLX_J(3, 1) VLX_J(3, 2) VLX_J(3, 3) VLX_J(3, 4) VLX_J(3, 5)
        VLX_J(4, 0) VLX_J(4, 1) VLX_J(4, 2) VLX_J(4, 3) VLX_J(4, 4)
        VLX_J(5, 0) VLX_J(5, 1) VLX_J(5, 2) VLX_J(5, 3)
        VLX_J(6, 0) VLX_J(6, 1) VLX_J(6, 2)
#undef VLX_J
    }
}
