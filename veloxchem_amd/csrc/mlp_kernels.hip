// Per atom-pair density network of the learned SCF guess, on the gfx950 matrix
// cores: n_in -> n_hidden -> n_hidden -> n_out with SiLU, BF16 weights and
// activations, FP32 accumulation, FP32 master weights and Adam.
//
// No reference counterpart: the reference starts every SCF from the SAD
// guess (src/pymodule/sadguessdriver.py:841-971); this network predicts the
// starting density block by block, and SAD stays the fallback.
//
// GEMM: C[M][N] = sum_k op(A)[m][k] op(B)[k][n], op(A) = A (M x K row-major)
// or A^T (A stored K x M), op(B) = B (K x N) or B^T (B stored N x K).  A
// 256-thread block owns a 64 x 64 tile of C; each wavefront a 32 x 32
// quarter, as 2 x 2 v_mfma_f32_16x16x32_bf16 tiles.  K advances by 32: the
// block stages op(A) as [m][k] and op(B) as [n][k] (k contiguous) in LDS, so
// that every lane reads its 8 consecutive k of one row or column with one
// 16-byte LDS load.  Every thread stages 8 elements of each operand with one 16-byte load (the
// leading dimensions of the bf16 buffers are multiples of 8; a group that crosses the edge of the
// matrix goes element by element), the next step's loads being issued before the products of this
// one.  Out-of-range rows, columns and k are staged as zeros.
//
// Weight gradients (K = batch) have few tiles: 16 of 64 x 64 for a 256 x 256 layer, on 256 CUs, each
// with a serial loop over the batch.  They are split over the batch (blockIdx.z), every part writing
// its own copy of the packed gradient, which one kernel then sums in a fixed order together with the
// bias gradients' parts.  With that, the wide staging loads and the gradient's way to the host through
// pinned memory, loss and gradient of a batch of 2048 (70-256-256-196) take 0.26 ms instead of 2.42;
// launches, the copy of the 0.5 MB gradient and the host's wait are most of what is left.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>

#include "../../include/vlxfock.h"
#include "../../include/vlxguess.h"
#include "vlx_types.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

namespace {

// BF16 as its 16 bits; conversions round to nearest even (finite inputs)
__host__ __device__ __forceinline__ uint16_t f2bf(float x)
{
    uint32_t u;
    std::memcpy(&u, &x, 4);
    u += 0x7fffu + ((u >> 16) & 1u);
    return static_cast<uint16_t>(u >> 16);
}
[[maybe_unused]] __host__ __device__ __forceinline__ float bf2f(uint16_t h)
{
    const uint32_t u = static_cast<uint32_t>(h) << 16;
    float x;
    std::memcpy(&x, &u, 4);
    return x;
}

__device__ __forceinline__ float sigmoid(float x) { return 1.0f / (1.0f + __expf(-x)); }

constexpr int TILE = 64;
constexpr int KT = 32;
constexpr int LDS_ROW = KT + 8;  // bf16 per staged row (padding against bank conflicts)

enum Epilogue {
    EPI_STORE = 0,       // C (fp32), part blockIdx.z at out_f + blockIdx.z * part_stride
    EPI_BIAS = 1,        // C + bias (fp32)
    EPI_BIAS_SILU = 2,   // H = C + bias (fp32) and silu(H) (bf16)
    EPI_SILU_GRAD = 3    // dH = C silu'(H) with H given (fp32 and bf16)
};

struct GemmArgs {
    const uint16_t* A;
    const uint16_t* B;
    int lda, ldb;        // leading dimensions as stored, multiples of 8
    int M, N, K;
    int kpart;           // k per part (multiple of KT); K: one part
    const float* bias;   // EPI_BIAS, EPI_BIAS_SILU
    const float* H;      // EPI_SILU_GRAD: pre-activations, M x N
    float* out_f;        // M x N fp32
    uint16_t* out_b;     // bf16, leading dimension ldo (EPI_BIAS_SILU, EPI_SILU_GRAD)
    int ldo;
    size_t part_stride;  // EPI_STORE
};

// 8 elements x[i0 .. i0 + 7] of a row of n valid ones as one 16-byte load, zeros past n.
__device__ __forceinline__ uint4 load8(const uint16_t* __restrict__ x, int i0, int n)
{
    if (i0 + 8 <= n) return *reinterpret_cast<const uint4*>(x + i0);
    union {
        uint16_t h[8];
        uint4 v;
    } u;
#pragma unroll
    for (int i = 0; i < 8; i++) u.h[i] = i0 + i < n ? x[i0 + i] : 0;
    return u.v;
}

// One thread's 8 elements of an operand's 64 x 32 step.  KMAJOR: stored [k][row], the thread takes
// 8 rows of one k; else stored [row][k], 8 consecutive k of one row.
template <bool KMAJOR>
__device__ __forceinline__ uint4 stage_load(const uint16_t* __restrict__ X, int ld, int r0, int nrow, int k0, int kend, int tid)
{
    const uint4 zero = {0, 0, 0, 0};
    if (KMAJOR) {
        const int k = k0 + (tid >> 3);
        return k < kend ? load8(X + (size_t)k * ld, r0 + (tid & 7) * 8, nrow) : zero;
    }
    const int r = r0 + (tid >> 2);
    return r < nrow ? load8(X + (size_t)r * ld, k0 + (tid & 3) * 8, kend) : zero;
}

template <bool KMAJOR>
__device__ __forceinline__ void stage_store(uint16_t* __restrict__ s, const uint4 v, int tid)
{
    if (KMAJOR) {
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 8; i++)
            s[((tid & 7) * 8 + i) * LDS_ROW + (tid >> 3)] = static_cast<uint16_t>(w[i >> 1] >> (16 * (i & 1)));
    } else {
        *reinterpret_cast<uint4*>(&s[(tid >> 2) * LDS_ROW + (tid & 3) * 8]) = v;
    }
}

template <bool TA, bool TB, int EPI>
__global__ void __launch_bounds__(256) mlp_gemm_kernel(const GemmArgs g)
{
    __shared__ __attribute__((aligned(16))) uint16_t sa[TILE * LDS_ROW];
    __shared__ __attribute__((aligned(16))) uint16_t sb[TILE * LDS_ROW];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int m0 = blockIdx.y * TILE, n0 = blockIdx.x * TILE;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;  // the wave's quarter of the tile
    const int kbeg = blockIdx.z * g.kpart, kend = min(g.K, kbeg + g.kpart);
    floatx4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    // A^T is stored [k][m], B without transpose [k][n]
    uint4 va = stage_load<TA>(g.A, g.lda, m0, g.M, kbeg, kend, tid);
    uint4 vb = stage_load<!TB>(g.B, g.ldb, n0, g.N, kbeg, kend, tid);
    for (int k0 = kbeg; k0 < kend; k0 += KT) {
        stage_store<TA>(sa, va, tid);
        stage_store<!TB>(sb, vb, tid);
        __syncthreads();
        if (k0 + KT < kend) {
            va = stage_load<TA>(g.A, g.lda, m0, g.M, k0 + KT, kend, tid);
            vb = stage_load<!TB>(g.B, g.ldb, n0, g.N, k0 + KT, kend, tid);
        }
        // lane l: row (or column) l % 16 of a 16-wide tile, k = 8 (l / 16) .. + 7
        const int fr = lane & 15, fk = (lane >> 4) * 8;
        bf16x8 af[2], bfr[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            af[i] = *reinterpret_cast<const bf16x8*>(&sa[(wm + 16 * i + fr) * LDS_ROW + fk]);
            bfr[i] = *reinterpret_cast<const bf16x8*>(&sb[(wn + 16 * i + fr) * LDS_ROW + fk]);
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bfr[j], acc[i][j], 0, 0, 0);
        __syncthreads();
    }
    // D of a 16 x 16 tile: lane l holds rows 4 (l / 16) + r, r = 0..3, of column l % 16
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int gm = m0 + wm + 16 * i + 4 * (lane >> 4) + r;
                const int gn = n0 + wn + 16 * j + (lane & 15);
                if (gm >= g.M || gn >= g.N) continue;
                const size_t o = (size_t)gm * g.N + gn;
                float v = acc[i][j][r];
                if (EPI == EPI_STORE) {
                    g.out_f[blockIdx.z * g.part_stride + o] = v;
                } else if (EPI == EPI_BIAS) {
                    g.out_f[o] = v + g.bias[gn];
                } else if (EPI == EPI_BIAS_SILU) {
                    v += g.bias[gn];
                    g.out_f[o] = v;
                    g.out_b[(size_t)gm * g.ldo + gn] = f2bf(v * sigmoid(v));
                } else {
                    const float h = g.H[o], s = sigmoid(h);
                    const float d = v * s * (1.0f + h * (1.0f - s));
                    g.out_f[o] = d;
                    g.out_b[(size_t)gm * g.ldo + gn] = f2bf(d);
                }
            }
}

// rows x cols fp32 to bf16 with leading dimension ld
__global__ void to_bf16_kernel(const float* __restrict__ x, uint16_t* __restrict__ y, size_t n, int cols, int ld)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        y[i / cols * ld + i % cols] = f2bf(x[i]);
}

// Per-sample mean squared error over the valid entries of a block (rows < ni, columns < nj of
// a block_cols-wide flattening), averaged over the m samples:
//   loss = (1/m) sum_s (1/(ni nj)) sum_valid (y - t)^2,  dY = 2 (y - t) / (m ni nj) (0 elsewhere).
__global__ void loss_grad_kernel(const float* __restrict__ y, const float* __restrict__ t,
                                 const int2* __restrict__ shape, int m, int n_out, int block_cols,
                                 float* __restrict__ dy_f, uint16_t* __restrict__ dy_b, int ldb,
                                 float* __restrict__ loss)
{
    float part = 0.f;
    const size_t total = (size_t)m * n_out;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const int s = static_cast<int>(i / n_out), o = static_cast<int>(i % n_out);
        const int2 sh = shape[s];
        float d = 0.f;
        if (o / block_cols < sh.x && o % block_cols < sh.y) {
            const float w = 1.0f / (static_cast<float>(m) * sh.x * sh.y);
            const float r = y[i] - t[i];
            part += r * r * w;
            d = 2.0f * r * w;
        }
        dy_f[i] = d;
        dy_b[(size_t)s * ldb + o] = f2bf(d);
    }
    for (int off = 32; off > 0; off >>= 1) part += __shfl_xor(part, off, 64);
    if ((threadIdx.x & 63) == 0) atomicAdd(loss, part);
}

// Column sums over the rows of part blockIdx.y of the three layers' fp32 gradients (bias gradients),
// layer blockIdx.z, into that part's copy of the packed gradient.  64 columns a block, 4 rows at a
// time: one block that loops over the whole batch is a serial chain of 2048 loads.
struct ColsumArgs {
    const float* x[3];
    int n[3];
    float* out[3];       // part 0 of the bias gradient
    int m, rows;         // rows in all, rows per part
    size_t part_stride;
};
__global__ void __launch_bounds__(256) colsum_kernel(const ColsumArgs g)
{
    __shared__ float part[4][64];
    const int l = blockIdx.z, n = g.n[l], c = blockIdx.x * 64 + (threadIdx.x & 63), q = threadIdx.x >> 6;
    const int r1 = min(g.m, static_cast<int>(blockIdx.y + 1) * g.rows);
    float s = 0.f;
    if (c < n)
        for (int r = blockIdx.y * g.rows + q; r < r1; r += 4) s += g.x[l][(size_t)r * n + c];
    part[q][threadIdx.x & 63] = s;
    __syncthreads();
    if (q == 0 && c < n) {
        const int t = threadIdx.x;
        g.out[l][blockIdx.y * g.part_stride + c] = (part[0][t] + part[1][t]) + (part[2][t] + part[3][t]);
    }
}

// sum of the parts of the packed gradient
__global__ void sum_parts_kernel(const float* __restrict__ parts, int nparts, size_t n, float* __restrict__ out)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        float s = parts[i];
        for (int p = 1; p < nparts; p++) s += parts[p * n + i];
        out[i] = s;
    }
}

// Adam on fp32 master weights, with their bf16 copies refreshed (bias vectors have no copy)
__global__ void adam_kernel(float* __restrict__ w, uint16_t* __restrict__ wb, const float* __restrict__ grad,
                            float* __restrict__ mom, float* __restrict__ vel, size_t n, int cols, int ld, float lr,
                            float b1, float b2, float eps, float c1, float c2)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const float gi = grad[i];
        const float mi = b1 * mom[i] + (1.0f - b1) * gi;
        const float vi = b2 * vel[i] + (1.0f - b2) * gi * gi;
        mom[i] = mi;
        vel[i] = vi;
        const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
        w[i] = wi;
        if (wb) wb[i / cols * ld + i % cols] = f2bf(wi);
    }
}

__global__ void clear_kernel(float* __restrict__ p, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.f;
}

int mfail(int code, const char* msg)
{
    vlx_set_last_error(msg);
    return code;
}

}  // namespace

// Layer l (0..2): W_l (fan_in x fan_out, row-major) and b_l (fan_out).
struct vlx_mlp {
    int device = 0;
    hipStream_t stream = nullptr;
    int n_in = 0, n_hidden = 0, n_out = 0, max_batch = 0, block_cols = 1;
    int fan_in[3], fan_out[3];
    size_t woff[3], boff[3], nparams = 0;  // offsets into the packed parameter vector
    float* p = nullptr;      // packed W0, b0, W1, b1, W2, b2 (fp32 master)
    float* grad = nullptr;   // same packing
    float* mom = nullptr;
    float* vel = nullptr;
    float* parts = nullptr;  // copies of the packed gradient, one per part of the batch
    float* h_grad = nullptr; // pinned: the gradient on its way to the caller
    uint16_t* wb[3] = {};    // bf16 copies of the weight matrices, leading dimension pad8(fan_out)
    int step = 0;
    // activations of one batch
    uint16_t *xb = nullptr, *a1b = nullptr, *a2b = nullptr, *dyb = nullptr, *dh2b = nullptr, *dh1b = nullptr;
    float *h1 = nullptr, *h2 = nullptr, *dyf = nullptr, *dh2f = nullptr, *dh1f = nullptr, *loss = nullptr;
};

namespace {

// Leading dimension of a bf16 buffer: rows start at 16-byte boundaries.
int pad8(int x) { return (x + 7) / 8 * 8; }

// Parts of a batch of m samples in the weight gradients, and samples per part: some 128 each (4 of
// the GEMM's k steps), at most MAX_PARTS.
constexpr int MAX_PARTS = 16;
int batch_parts(int m, int* rows)
{
    const int p = std::max(1, std::min(MAX_PARTS, m / 128));
    *rows = ((m + p - 1) / p + KT - 1) / KT * KT;
    return (m + *rows - 1) / *rows;
}

template <typename T>
hipError_t dalloc(T** p, size_t n)
{
    return hipMalloc(reinterpret_cast<void**>(p), std::max<size_t>(n, 1) * sizeof(T));
}

#define MLP_TRY(expr)                                                                   \
    do {                                                                                \
        hipError_t e_ = (expr);                                                         \
        if (e_ != hipSuccess) return mfail(VLX_ERR_HIP, hipGetErrorString(e_));         \
    } while (0)

template <bool TA, bool TB, int EPI>
int gemm(hipStream_t s, const GemmArgs& g, int parts = 1)
{
    if (g.M <= 0 || g.N <= 0 || g.K <= 0) return VLX_OK;
    dim3 grid((g.N + TILE - 1) / TILE, (g.M + TILE - 1) / TILE, parts);
    hipLaunchKernelGGL((mlp_gemm_kernel<TA, TB, EPI>), grid, dim3(256), 0, s, g);
    MLP_TRY(hipGetLastError());
    return VLX_OK;
}

int grid_for(size_t n) { return static_cast<int>(std::min<size_t>((n + 255) / 256, 4096)); }

int forward(vlx_mlp* net, const float* d_x, int m, float* d_y)
{
    hipStream_t s = net->stream;
    const int H = net->n_hidden, ldx = pad8(net->n_in), ldh = pad8(H), ldy = pad8(net->n_out);
    to_bf16_kernel<<<grid_for((size_t)m * net->n_in), 256, 0, s>>>(d_x, net->xb, (size_t)m * net->n_in, net->n_in, ldx);
    MLP_TRY(hipGetLastError());
    GemmArgs g{};
    g = {net->xb, net->wb[0], ldx, ldh, m, H, net->n_in, net->n_in, net->p + net->boff[0], nullptr, net->h1, net->a1b, ldh, 0};
    int rc = gemm<false, false, EPI_BIAS_SILU>(s, g);
    if (rc) return rc;
    g = {net->a1b, net->wb[1], ldh, ldh, m, H, H, H, net->p + net->boff[1], nullptr, net->h2, net->a2b, ldh, 0};
    rc = gemm<false, false, EPI_BIAS_SILU>(s, g);
    if (rc) return rc;
    g = {net->a2b, net->wb[2], ldh, ldy, m, net->n_out, H, H, net->p + net->boff[2], nullptr, d_y, nullptr, 0, 0};
    return gemm<false, false, EPI_BIAS>(s, g);
}

}  // namespace

extern "C" {

int vlx_mlp_create(vlx_context* ctx, int n_in, int n_hidden, int n_out, int block_cols, int max_batch, vlx_mlp** out)
{
    if (!ctx || !out) return mfail(VLX_ERR_ARG, "NULL argument to vlx_mlp_create");
    if (n_in <= 0 || n_hidden <= 0 || n_out <= 0 || max_batch <= 0 || block_cols <= 0)
        return mfail(VLX_ERR_ARG, "vlx_mlp_create: sizes must be positive");
    auto net = new vlx_mlp();
    net->stream = static_cast<hipStream_t>(vlx_context_stream(ctx));
    MLP_TRY(hipGetDevice(&net->device));
    net->n_in = n_in;
    net->n_hidden = n_hidden;
    net->n_out = n_out;
    net->block_cols = block_cols;
    net->max_batch = max_batch;
    const int fi[3] = {n_in, n_hidden, n_hidden}, fo[3] = {n_hidden, n_hidden, n_out};
    size_t off = 0;
    for (int l = 0; l < 3; l++) {
        net->fan_in[l] = fi[l];
        net->fan_out[l] = fo[l];
        net->woff[l] = off;
        off += (size_t)fi[l] * fo[l];
        net->boff[l] = off;
        off += fo[l];
    }
    net->nparams = off;
    const size_t mb = static_cast<size_t>(max_batch);
    hipError_t e = hipSuccess;
    for (float** q : {&net->p, &net->grad, &net->mom, &net->vel})
        if (e == hipSuccess) e = dalloc(q, off);
    // batch_parts takes no more for any batch up to max_batch
    const int max_parts = std::max(1, std::min(MAX_PARTS, max_batch / 128));
    if (e == hipSuccess) e = dalloc(&net->parts, off * max_parts);
    if (e == hipSuccess) e = hipHostMalloc(reinterpret_cast<void**>(&net->h_grad), (off + 1) * sizeof(float));
    for (int l = 0; l < 3 && e == hipSuccess; l++) e = dalloc(&net->wb[l], (size_t)fi[l] * pad8(fo[l]));
    if (e == hipSuccess) e = dalloc(&net->xb, mb * pad8(n_in));
    for (uint16_t** q : {&net->a1b, &net->a2b, &net->dh2b, &net->dh1b})
        if (e == hipSuccess) e = dalloc(q, mb * pad8(n_hidden));
    if (e == hipSuccess) e = dalloc(&net->dyb, mb * pad8(n_out));
    for (float** q : {&net->h1, &net->h2, &net->dh2f, &net->dh1f})
        if (e == hipSuccess) e = dalloc(q, mb * n_hidden);
    if (e == hipSuccess) e = dalloc(&net->dyf, mb * n_out);
    if (e == hipSuccess) e = dalloc(&net->loss, 1);
    if (e != hipSuccess) {
        vlx_mlp_destroy(net);
        return mfail(VLX_ERR_NOMEM, "vlx_mlp_create: device allocation failed");
    }
    *out = net;
    return VLX_OK;
}

void vlx_mlp_destroy(vlx_mlp* net)
{
    if (!net) return;
    if (net->stream) (void)hipStreamSynchronize(net->stream);
    if (net->h_grad) (void)hipHostFree(net->h_grad);
    for (float* q : {net->p, net->grad, net->parts, net->mom, net->vel, net->h1, net->h2, net->dyf, net->dh2f, net->dh1f, net->loss})
        if (q) (void)hipFree(q);
    for (uint16_t* q : {net->wb[0], net->wb[1], net->wb[2], net->xb, net->a1b, net->a2b, net->dyb, net->dh2b, net->dh1b})
        if (q) (void)hipFree(q);
    delete net;
}

int vlx_mlp_num_params(vlx_mlp* net, long long* n)
{
    if (!net || !n) return mfail(VLX_ERR_ARG, "NULL argument");
    *n = static_cast<long long>(net->nparams);
    return VLX_OK;
}

int vlx_mlp_set_params(vlx_mlp* net, const float* params)
{
    if (!net || !params) return mfail(VLX_ERR_ARG, "NULL argument");
    MLP_TRY(hipMemcpyAsync(net->p, params, net->nparams * sizeof(float), hipMemcpyHostToDevice, net->stream));
    for (int l = 0; l < 3; l++) {
        const size_t n = (size_t)net->fan_in[l] * net->fan_out[l];
        to_bf16_kernel<<<grid_for(n), 256, 0, net->stream>>>(net->p + net->woff[l], net->wb[l], n, net->fan_out[l],
                                                             pad8(net->fan_out[l]));
        MLP_TRY(hipGetLastError());
    }
    // a fresh parameter set restarts the optimiser
    clear_kernel<<<(int)((net->nparams + 255) / 256), 256, 0, net->stream>>>(net->mom, (int)net->nparams);
    clear_kernel<<<(int)((net->nparams + 255) / 256), 256, 0, net->stream>>>(net->vel, (int)net->nparams);
    MLP_TRY(hipGetLastError());
    net->step = 0;
    MLP_TRY(hipStreamSynchronize(net->stream));
    return VLX_OK;
}

int vlx_mlp_get_params(vlx_mlp* net, float* params)
{
    if (!net || !params) return mfail(VLX_ERR_ARG, "NULL argument");
    MLP_TRY(hipMemcpyAsync(params, net->p, net->nparams * sizeof(float), hipMemcpyDeviceToHost, net->stream));
    MLP_TRY(hipStreamSynchronize(net->stream));
    return VLX_OK;
}

int vlx_mlp_forward(vlx_mlp* net, const float* d_x, int m, float* d_y)
{
    if (!net || !d_x || !d_y) return mfail(VLX_ERR_ARG, "NULL argument");
    if (m < 0 || m > net->max_batch) return mfail(VLX_ERR_ARG, "vlx_mlp_forward: batch outside 0..max_batch");
    return forward(net, d_x, m, d_y);
}

int vlx_mlp_loss_grad(vlx_mlp* net, const float* d_x, const float* d_target, const int* d_shape, int m, float* d_y,
                      float* loss, float* grads)
{
    if (!net || !d_x || !d_target || !d_shape || !d_y || !loss) return mfail(VLX_ERR_ARG, "NULL argument");
    if (m <= 0 || m > net->max_batch) return mfail(VLX_ERR_ARG, "vlx_mlp_loss_grad: batch outside 1..max_batch");
    hipStream_t s = net->stream;
    int rc = forward(net, d_x, m, d_y);
    if (rc) return rc;
    clear_kernel<<<1, 64, 0, s>>>(net->loss, 1);
    const size_t ny = (size_t)m * net->n_out;
    const int H = net->n_hidden, NO = net->n_out, ldx = pad8(net->n_in), ldh = pad8(H), ldy = pad8(NO);
    loss_grad_kernel<<<grid_for(ny), 256, 0, s>>>(d_y, d_target, reinterpret_cast<const int2*>(d_shape), m, NO,
                                                   net->block_cols, net->dyf, net->dyb, ldy, net->loss);
    MLP_TRY(hipGetLastError());
    int rows = 0;
    const int parts = batch_parts(m, &rows);
    float* gw[3] = {net->parts + net->woff[0], net->parts + net->woff[1], net->parts + net->woff[2]};
    GemmArgs g{};
    // layer 3: dW2 = A2^T dY, dH2 = (dY W2^T) silu'(H2)
    g = {net->a2b, net->dyb, ldh, ldy, H, NO, m, rows, nullptr, nullptr, gw[2], nullptr, 0, net->nparams};
    if ((rc = gemm<true, false, EPI_STORE>(s, g, parts))) return rc;
    g = {net->dyb, net->wb[2], ldy, ldy, m, H, NO, NO, nullptr, net->h2, net->dh2f, net->dh2b, ldh, 0};
    if ((rc = gemm<false, true, EPI_SILU_GRAD>(s, g))) return rc;
    // layer 2: dW1 = A1^T dH2, dH1 = (dH2 W1^T) silu'(H1)
    g = {net->a1b, net->dh2b, ldh, ldh, H, H, m, rows, nullptr, nullptr, gw[1], nullptr, 0, net->nparams};
    if ((rc = gemm<true, false, EPI_STORE>(s, g, parts))) return rc;
    g = {net->dh2b, net->wb[1], ldh, ldh, m, H, H, H, nullptr, net->h1, net->dh1f, net->dh1b, ldh, 0};
    if ((rc = gemm<false, true, EPI_SILU_GRAD>(s, g))) return rc;
    // layer 1: dW0 = X^T dH1
    g = {net->xb, net->dh1b, ldx, ldh, net->n_in, H, m, rows, nullptr, nullptr, gw[0], nullptr, 0, net->nparams};
    if ((rc = gemm<true, false, EPI_STORE>(s, g, parts))) return rc;
    // bias gradients, then the sum of the parts
    const ColsumArgs cs{{net->dh1f, net->dh2f, net->dyf}, {H, H, NO},
                        {net->parts + net->boff[0], net->parts + net->boff[1], net->parts + net->boff[2]},
                        m, rows, net->nparams};
    colsum_kernel<<<dim3((std::max(H, NO) + 63) / 64, parts, 3), 256, 0, s>>>(cs);
    sum_parts_kernel<<<grid_for(net->nparams), 256, 0, s>>>(net->parts, parts, net->nparams, net->grad);
    MLP_TRY(hipGetLastError());
    // through pinned memory: a copy into the caller's pageable array would be staged by the runtime
    float* h_loss = net->h_grad + net->nparams;
    MLP_TRY(hipMemcpyAsync(h_loss, net->loss, sizeof(float), hipMemcpyDeviceToHost, s));
    if (grads) MLP_TRY(hipMemcpyAsync(net->h_grad, net->grad, net->nparams * sizeof(float), hipMemcpyDeviceToHost, s));
    MLP_TRY(hipStreamSynchronize(s));
    *loss = *h_loss;
    if (grads) std::memcpy(grads, net->h_grad, net->nparams * sizeof(float));
    return VLX_OK;
}

int vlx_mlp_adam_step(vlx_mlp* net, float lr, float beta1, float beta2, float eps)
{
    if (!net) return mfail(VLX_ERR_ARG, "NULL argument");
    net->step++;
    const float c1 = 1.0f - std::pow(beta1, static_cast<float>(net->step));
    const float c2 = 1.0f - std::pow(beta2, static_cast<float>(net->step));
    for (int l = 0; l < 3; l++) {
        const size_t nw = (size_t)net->fan_in[l] * net->fan_out[l];
        adam_kernel<<<grid_for(nw), 256, 0, net->stream>>>(net->p + net->woff[l], net->wb[l], net->grad + net->woff[l],
                                                          net->mom + net->woff[l], net->vel + net->woff[l], nw,
                                                          net->fan_out[l], pad8(net->fan_out[l]), lr, beta1, beta2,
                                                          eps, c1, c2);
        const size_t nb = net->fan_out[l];
        adam_kernel<<<grid_for(nb), 256, 0, net->stream>>>(net->p + net->boff[l], nullptr, net->grad + net->boff[l],
                                                          net->mom + net->boff[l], net->vel + net->boff[l], nb, 1, 1,
                                                          lr, beta1, beta2, eps, c1, c2);
    }
    MLP_TRY(hipGetLastError());
    return VLX_OK;
}

}  // extern "C"
