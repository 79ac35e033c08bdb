// Surrogate closure network of libbrownian: a multilayer perceptron
//   144 -> 256 -> 256 -> 256 -> 12, SiLU hidden activations,
// run and trained on the GPU with its own kernels.  Matrix products use the
// gfx950 matrix cores (V_MFMA_F32_32X32X16_BF16: BF16 operands, FP32
// accumulation, operands staged through LDS); weights are kept in FP32 (Adam
// state too) with BF16 copies for the products.  The output is the per-interval colloid impulse mean (6)
// and log-variance (6) in standardised units; the loss is the Gaussian
// negative log-likelihood.
//
// Padded shapes (multiples of 32): input 144 -> 160 (zero columns), output
// 12 -> 32 (zero weight columns).  Batch rows are padded to 32 with zeros.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <string.h>

#include <cmath>
#include <type_traits>
#include <string>
#include <mutex>
#include <vector>

#include "../../include/brownian.h"
#include "mlp.h"

namespace bw {

typedef float f32x16 __attribute__((ext_vector_type(16)));

// FP32 -> BF16, round to nearest even (NaN kept quiet)
__device__ __forceinline__ unsigned short f2bf(float f) {
    unsigned u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u) return (unsigned short)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// One 64 x 64 block of C (M x N) = op(A) (M x K) . op(B) (K x N) on the gfx950
// matrix cores (V_MFMA_F32_32X32X16_BF16: BF16 operands, FP32 accumulation), by
// four waves, each a 32 x 32 quadrant (acc).  K goes through LDS in stages of
// 128; a stage's global loads (128 bits, eight in flight per thread) are sent
// before the last stage is multiplied, so that a product of K <= 256 waits for
// memory twice.  A transposed operand is transposed on its way into LDS, two k
// at a time.  M, N and K are multiples of 32; rows or columns of a block past M
// or N are zero-filled.
//   TA = 0: A is M x K row-major (lda = row stride); TA = 1: A is stored K x M.
//   TB = 0: B is K x N row-major;                    TB = 1: B is stored N x K.
// Operand layout of one 32x32x16 product: lane l supplies A[l%32][k] and
// B[k][l%32] for 8 values of k selected by l/32 (the same selection for A and
// B, so that the sum over k does not depend on it); accumulator element i of
// lane l is C[8(i/4) + 4(l/32) + i%4][l%32].
constexpr int GEMM_B = 64, GEMM_KS = 128;
// place of element (row, k) of a stage: rows of 128 BF16 without padding, their
// 16-byte granules permuted by the row so that both the reads (a granule of 16
// consecutive rows) and the transposed writes (one k of every eighth row) spread
// over the banks
__device__ __forceinline__ int gemm_place(int row, int k) {
    return row * GEMM_KS + ((((k >> 3) ^ row ^ (row >> 3)) & 15) << 3) + (k & 7);
}
template <int T>
__device__ __forceinline__ void gemm_load(const unsigned short *__restrict__ A, int M, int K, int lda, int m0, int k0,
                                          u32x4 *v) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        int row, k;
        if (T == 0) {  // a row's granule
            const int id = threadIdx.x + 256 * i;
            row = id >> 4;
            k = k0 + (id & 15) * 8;
        } else {  // eight rows of one k; v[2j], v[2j + 1] are neighbouring k
            const int id = threadIdx.x + 256 * (i >> 1);
            row = (id & 7) * 8;
            k = k0 + (id >> 3) * 2 + (i & 1);
        }
        v[i] = u32x4{0u, 0u, 0u, 0u};
        if (m0 + row < M && k < K)
            v[i] = *(const u32x4 *)(T == 0 ? A + (size_t)(m0 + row) * lda + k : A + (size_t)k * lda + m0 + row);
    }
}
template <int T>
__device__ __forceinline__ void gemm_store(unsigned short *s, const u32x4 *v) {
    if (T == 0) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int id = threadIdx.x + 256 * i;
            *(u32x4 *)(s + gemm_place(id >> 4, (id & 15) * 8)) = v[i];
        }
    } else {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int id = threadIdx.x + 256 * i, row = (id & 7) * 8, k = (id >> 3) * 2;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const unsigned a = (v[2 * i][j >> 1] >> (16 * (j & 1))) & 0xffffu;
                const unsigned b = (v[2 * i + 1][j >> 1] >> (16 * (j & 1))) & 0xffffu;
                *(unsigned *)(s + gemm_place(row + j, k)) = a | (b << 16);
            }
        }
    }
}
template <int TA, int TB>
__device__ __forceinline__ f32x16 gemm_block(const unsigned short *__restrict__ A, const unsigned short *__restrict__ B, int M,
                                             int N, int K, int lda, int ldb, int m0, int n0, unsigned short *smem) {
    unsigned short *As = smem, *Bs = smem + GEMM_B * GEMM_KS;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int ra = (w >> 1) * 32 + (lane & 31), rb = (w & 1) * 32 + (lane & 31), kh = (lane >> 5) * 8;
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; i++) acc[i] = 0.0f;
    u32x4 va[4], vb[4];
    gemm_load<TA>(A, M, K, lda, m0, 0, va);
    gemm_load<TB == 1 ? 0 : 1>(B, N, K, ldb, n0, 0, vb);
    for (int k0 = 0; k0 < K; k0 += GEMM_KS) {
        gemm_store<TA>(As, va);
        gemm_store<TB == 1 ? 0 : 1>(Bs, vb);
        __syncthreads();
        if (k0 + GEMM_KS < K) {
            gemm_load<TA>(A, M, K, lda, m0, k0 + GEMM_KS, va);
            gemm_load<TB == 1 ? 0 : 1>(B, N, K, ldb, n0, k0 + GEMM_KS, vb);
        }
#pragma unroll
        for (int kk = 0; kk < GEMM_KS; kk += 16) {  // (past K both operands are zero)
            const u32x4 a = *(const u32x4 *)(As + gemm_place(ra, kk + kh));
            const u32x4 b = *(const u32x4 *)(Bs + gemm_place(rb, kk + kh));
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                          acc, 0, 0, 0);
        }
        __syncthreads();
    }
    return acc;
}
// f(m, n, value) for this thread's elements of the block at (m0, n0)
template <class F>
__device__ __forceinline__ void gemm_elements(const f32x16 &acc, int M, int N, int m0, int n0, F &&f) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int m1 = m0 + (w >> 1) * 32, n = n0 + (w & 1) * 32 + (lane & 31);
    if (m1 >= M || n >= N) return;
#pragma unroll
    for (int i = 0; i < 16; i++) f(m1 + (i >> 2) * 8 + (lane >> 5) * 4 + (i & 3), n, acc[i]);
}

// one hidden layer: Z = X W + b (kept for the backward pass when Z is not
// null), Hb = bf16(silu(Z))
__global__ __launch_bounds__(256) void k_layer(const unsigned short *__restrict__ X, const unsigned short *__restrict__ W,
                                               const float *__restrict__ bias, int M, int N, int K, float *__restrict__ Z,
                                               unsigned short *__restrict__ Hb) {
    __shared__ __align__(16) unsigned short s[2 * GEMM_B * GEMM_KS];
    const int nbn = (N + GEMM_B - 1) / GEMM_B;
    const int m0 = (blockIdx.x / nbn) * GEMM_B, n0 = (blockIdx.x % nbn) * GEMM_B;
    const f32x16 acc = gemm_block<0, 0>(X, W, M, N, K, K, N, m0, n0, s);
    gemm_elements(acc, M, N, m0, n0, [&](int m, int n, float v) {
        const float z = v + bias[n];
        const float h = z / (1.0f + expf(-z));
        if (Z) Z[(size_t)m * N + n] = z;
        Hb[(size_t)m * N + n] = f2bf(h);
    });
}
// the output layer: Y = X W + b; rows not null: its first n rows without their
// padding, n x MLP_OUT, in place of Y
__global__ __launch_bounds__(256) void k_layer_out(const unsigned short *__restrict__ X, const unsigned short *__restrict__ W,
                                                   const float *__restrict__ bias, int M, float *__restrict__ Y,
                                                   float *__restrict__ rows, int n_rows) {
    __shared__ __align__(16) unsigned short s[2 * GEMM_B * GEMM_KS];
    const f32x16 acc = gemm_block<0, 0>(X, W, M, MLP_OUTP, MLP_H, MLP_H, MLP_OUTP, blockIdx.x * GEMM_B, 0, s);
    gemm_elements(acc, M, MLP_OUTP, blockIdx.x * GEMM_B, 0, [&](int m, int n, float v) {
        if (!rows) Y[(size_t)m * MLP_OUTP + n] = v + bias[n];
        else if (m < n_rows && n < MLP_OUT) rows[(size_t)m * MLP_OUT + n] = v + bias[n];
    });
}

__global__ void k_to_bf16(const float *__restrict__ x, unsigned short *__restrict__ y, long long n) {
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = f2bf(x[i]);
}

// standardised, padded BF16 input rows: xb[i][f] = bf16((x[idx[i]][f] - mean[f]) * istd[f])
__global__ void k_mlp_input(const float *__restrict__ x, const int *__restrict__ idx, int n, int n_pad,
                            const float *__restrict__ mean, const float *__restrict__ istd,
                            unsigned short *__restrict__ xb) {
    long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (long long)n_pad * MLP_INP) return;
    const int i = (int)(e / MLP_INP), f = (int)(e - (long long)i * MLP_INP);
    float v = 0.0f;
    if (i < n && f < MLP_IN) {
        const long long row = idx ? idx[i] : i;
        v = (x[row * MLP_IN + f] - mean[f]) * istd[f];
    }
    xb[e] = f2bf(v);
}

// The output layer and the Gaussian NLL on standardised targets:
// loss = 0.5 sum_k (s_k + (t_k - mu_k)^2 e^{-s_k}) with mu = y[0:6], s = y[6:12]
// (clamped to +-20); gradients scaled by 1/n.  A block holds all 12 columns of
// its 64 rows: they meet in LDS, a thread per row.
__global__ __launch_bounds__(256) void k_layer_nll(const unsigned short *__restrict__ X, const unsigned short *__restrict__ W,
                                                   const float *__restrict__ bias, int M, const float *__restrict__ t,
                                                   const int *__restrict__ idx, int n, const float *__restrict__ tmean,
                                                   const float *__restrict__ tistd, float *__restrict__ dy,
                                                   unsigned short *__restrict__ dyb, float *__restrict__ loss) {
    __shared__ __align__(16) unsigned short s[2 * GEMM_B * GEMM_KS];
    __shared__ float s_y[GEMM_B][MLP_OUTP + 1];
    const int m0 = blockIdx.x * GEMM_B;
    const f32x16 acc = gemm_block<0, 0>(X, W, M, MLP_OUTP, MLP_H, MLP_H, MLP_OUTP, m0, 0, s);
    gemm_elements(acc, M, MLP_OUTP, m0, 0, [&](int m, int c, float v) { s_y[m - m0][c] = v + bias[c]; });
    __syncthreads();
    const int i = m0 + threadIdx.x;
    if (threadIdx.x < GEMM_B && i < M) {
        float *y = s_y[threadIdx.x];
        float g[MLP_OUT], l = 0.0f;
        for (int c = 0; c < MLP_OUT; c++) g[c] = 0.0f;
        if (i < n) {
            const long long row = idx ? idx[i] : i;
            const float inv_n = 1.0f / (float)n;
            for (int k = 0; k < MLP_T; k++) {
                const float tk = (t[row * MLP_T + k] - tmean[k]) * tistd[k];
                const float mu = y[k];
                const float sv = fminf(fmaxf(y[MLP_T + k], -20.0f), 20.0f);
                const float e = expf(-sv), d = tk - mu;
                l += 0.5f * (sv + d * d * e);
                g[k] = -d * e * inv_n;
                g[MLP_T + k] = 0.5f * (1.0f - d * d * e) * inv_n;
            }
            loss[i] = l;
        }
        for (int c = 0; c < MLP_OUTP; c++) y[c] = c < MLP_OUT ? g[c] : 0.0f;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < GEMM_B * MLP_OUTP; e += 256) {
        const int r = e / MLP_OUTP, c = e % MLP_OUTP;
        if (m0 + r >= M) break;
        const float g = s_y[r][c];
        dy[(size_t)(m0 + r) * MLP_OUTP + c] = g;
        dyb[(size_t)(m0 + r) * MLP_OUTP + c] = f2bf(g);
    }
}

// The backward pass of one layer, three independent products in one launch so
// that each fills what the others leave idle (a weight gradient alone is 12 to
// 16 blocks per split of the batch):
//  - the weight gradient X^T dZ (K x N), the batch split into np chunks of kc
//    rows, one partial product each;
//  - the bias gradient: column sums of dZ over blocks of COLSUM_ROWS rows;
//  - dZ of the layer below, (dZ W^T) silu'(Z) with silu'(z) = s (1 + z (1 - s)),
//    s = sigmoid(z) (not for the first layer: zbelow null).
// k_update adds the parts in order.
constexpr int COLSUM_ROWS = 128;
constexpr int WGRAD_SPLITS = 8;  // most chunks of the batch in a weight-gradient product
struct BackArgs {
    const unsigned short *x, *dzb, *w;  // input (rows x K), dZ (rows x N), weights (K x N)
    const float *dz, *zbelow;
    float *wpart, *bpart, *dzbelow;
    unsigned short *dzbbelow;
    int rows, K, N, np, kc;
};
__host__ __device__ inline int back_blocks(int m, int n) { return ((m + GEMM_B - 1) / GEMM_B) * ((n + GEMM_B - 1) / GEMM_B); }
__host__ __device__ inline int colsum_blocks(int rows, int n) { return ((n + 63) / 64) * ((rows + COLSUM_ROWS - 1) / COLSUM_ROWS); }
__global__ __launch_bounds__(256) void k_layer_back(BackArgs a) {
    __shared__ __align__(16) unsigned short s[2 * GEMM_B * GEMM_KS];
    int b = blockIdx.x;
    const int nh = a.zbelow ? back_blocks(a.rows, a.K) : 0, nw = a.np * back_blocks(a.K, a.N);
    if (b < nh) {  // first: the next launch waits for these
        const int nbn = (a.K + GEMM_B - 1) / GEMM_B, m0 = (b / nbn) * GEMM_B, n0 = (b % nbn) * GEMM_B;
        const f32x16 acc = gemm_block<0, 1>(a.dzb, a.w, a.rows, a.K, a.N, a.N, a.N, m0, n0, s);
        gemm_elements(acc, a.rows, a.K, m0, n0, [&](int m, int n, float v) {
            const size_t o = (size_t)m * a.K + n;
            const float zz = a.zbelow[o], sg = 1.0f / (1.0f + expf(-zz));
            const float g = v * (sg * (1.0f + zz * (1.0f - sg)));
            a.dzbelow[o] = g;
            a.dzbbelow[o] = f2bf(g);
        });
        return;
    }
    b -= nh;
    if (b < nw) {
        const int per = back_blocks(a.K, a.N), p = b / per, q = b % per, nbn = (a.N + GEMM_B - 1) / GEMM_B;
        const int m0 = (q / nbn) * GEMM_B, n0 = (q % nbn) * GEMM_B, k0 = p * a.kc;
        const f32x16 acc = gemm_block<1, 0>(a.x + (size_t)k0 * a.K, a.dzb + (size_t)k0 * a.N, a.K, a.N,
                                            min(a.kc, a.rows - k0), a.K, a.N, m0, n0, s);
        float *c = a.wpart + (size_t)p * a.K * a.N;
        gemm_elements(acc, a.K, a.N, m0, n0, [&](int m, int n, float v) { c[(size_t)m * a.N + n] = v; });
        return;
    }
    b -= nw;
    // four row phases per column, combined in order
    float(*sum)[64] = (float(*)[64])s;
    const int nc = (a.N + 63) / 64, y = b / nc, c = (b % nc) * 64 + (threadIdx.x & 63), ph = threadIdx.x >> 6;
    const int r0 = y * COLSUM_ROWS, r1 = min(a.rows, r0 + COLSUM_ROWS);
    float v = 0.0f;
    if (c < a.N)
        for (int r = r0 + ph; r < r1; r += 4) v += a.dz[(size_t)r * a.N + c];
    sum[ph][threadIdx.x & 63] = v;
    __syncthreads();
    if (threadIdx.x < 64 && c < a.N)
        a.bpart[(size_t)y * a.N + c] = ((sum[0][threadIdx.x] + sum[1][threadIdx.x]) + sum[2][threadIdx.x]) + sum[3][threadIdx.x];
}

// All parameters in one launch: the gradient as the sum of its np parts in
// order, then either stored in the logical layout (unpadded, W1, b1, ..., b4) or
// one step of Adam (Kingma & Ba, 2015) on the FP32 master weights, which also
// refreshes the BF16 copy.  Parameters outside the logical shape stay zero.
struct ParamSeg {
    float *w, *m, *v;
    unsigned short *wb;  // null for biases
    const float *part;
    int np, n, cols, lrows, lcols, first, lfirst;  // padded size and columns; logical; first element in either layout
};
struct ParamTable {
    ParamSeg s[2 * MLP_L];
    int total;
};
__device__ __forceinline__ const ParamSeg &param_seg(const ParamTable &t, int i) {
    int q = 0;
    while (q + 1 < 2 * MLP_L && i >= t.s[q + 1].first) q++;
    return t.s[q];
}
// place of element e of a segment in the logical layout, -1 for padding
__device__ __forceinline__ int param_logical(const ParamSeg &p, int e) {
    const int r = e / p.cols, c = e - r * p.cols;
    return r < p.lrows && c < p.lcols ? p.lfirst + r * p.lcols + c : -1;
}
__device__ __forceinline__ float param_grad(const ParamSeg &p, int e) {
    float a = 0.0f;
    for (int q = 0; q < p.np; q++) a += p.part[(size_t)q * p.n + e];
    return a;
}
__global__ void k_adam(ParamTable t, float lr, float b1, float b2, float c1, float c2, float eps) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= t.total) return;
    const ParamSeg &p = param_seg(t, i);
    const int e = i - p.first;
    const float gi = param_grad(p, e);
    const float mi = b1 * p.m[e] + (1.0f - b1) * gi;
    const float vi = b2 * p.v[e] + (1.0f - b2) * gi * gi;
    p.m[e] = mi;
    p.v[e] = vi;
    const float wi = p.w[e] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    p.w[e] = wi;
    if (p.wb) p.wb[e] = f2bf(wi);
}
// gradients (GRAD) or parameters in the logical layout
template <bool GRAD>
__global__ void k_pack(ParamTable t, float *__restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= t.total) return;
    const ParamSeg &p = param_seg(t, i);
    const int e = i - p.first, o = param_logical(p, e);
    if (o >= 0) out[o] = GRAD ? param_grad(p, e) : p.w[e];
}

// Activations of bw_mlp_forward_noalloc for up to NOALLOC_ROWS rows, in a
// file-scope device array instead of allocations: input (BF16), three hidden
// layers (BF16) and the padded output.  Each GPU holds its own copy until the process ends.
constexpr int NOALLOC_ROWS = 1024;
constexpr size_t NOALLOC_ROW_BYTES = (size_t)MLP_INP * 2 + (size_t)MLP_OUTP * 4 + 3 * ((size_t)MLP_H * 2);
static __device__ __align__(256) unsigned char scratch[NOALLOC_ROWS * NOALLOC_ROW_BYTES];

}  // namespace bw

using namespace bw;

// ------------------------------------------------------------------- host
struct bw_mlp {
    std::string err;
    hipStream_t st = nullptr;
    int K[MLP_L] = {MLP_INP, MLP_H, MLP_H, MLP_H};
    int N[MLP_L] = {MLP_H, MLP_H, MLP_H, MLP_OUTP};
    int Kl[MLP_L] = {MLP_IN, MLP_H, MLP_H, MLP_H};   // logical (unpadded)
    int Nl[MLP_L] = {MLP_H, MLP_H, MLP_H, MLP_OUT};
    float *W[MLP_L] = {}, *b[MLP_L] = {};
    float *packed = nullptr;  // parameters or gradients in the logical layout, on their way to the host
    float *mW[MLP_L] = {}, *vW[MLP_L] = {}, *mb[MLP_L] = {}, *vb[MLP_L] = {};
    unsigned short *Wb[MLP_L] = {};
    float *xmean = nullptr, *xistd = nullptr, *tmean = nullptr, *tistd = nullptr;
    long long adam_t = 0;
    MlpBuf tb;  // training / host-call activations
    unsigned char *scratch = nullptr;  // device address of the scratch array on the network's GPU
    // a host call's rows: 648 bytes for each of the largest call's, kept until
    // the network is destroyed, as its activations are (two hipMalloc and hipFree
    // a call otherwise)
    float *xin = nullptr, *tin = nullptr, *yout = nullptr;
    float *ypin = nullptr;    // outputs of up to PINNED_ROWS rows, in pinned host memory
    long long xin_rows = 0;
    // data set on the device, and the rows' losses
    float *dX = nullptr, *dT = nullptr, *dloss = nullptr;
    int *didx = nullptr;
    long long dn = 0;
    std::vector<void *> allocs;
};

namespace bw {
// floats of the partial weight and bias gradients of `rows` rows, layer by layer
static size_t part_floats(int rows, int l) {
    const size_t K = l == 0 ? MLP_INP : MLP_H, N = l == MLP_L - 1 ? MLP_OUTP : MLP_H;
    return WGRAD_SPLITS * K * N + ((size_t)rows / COLSUM_ROWS + 1) * N;
}
int mlp_buf_alloc(MlpBuf &b, int rows, bool train) {
    int cap = (rows + 31) / 32 * 32;
    if (cap <= b.cap && (b.part || !train)) return 0;
    cap = std::max(cap, b.cap);
    mlp_buf_free(b);
    auto al = [](auto **p, size_t n) {
        void *q = nullptr;
        if (hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(**p)) != hipSuccess) return 1;
        hipMemset(q, 0, std::max<size_t>(n, 1) * sizeof(**p));
        *p = (std::remove_reference_t<decltype(*p)>)q;
        return 0;
    };
    int bad = al(&b.Xb, (size_t)cap * MLP_INP) | al(&b.Y, (size_t)cap * MLP_OUTP);
    for (int l = 0; l < 3; l++) bad |= al(&b.Hb[l], (size_t)cap * MLP_H);
    if (train) {
        bad |= al(&b.dY, (size_t)cap * MLP_OUTP) | al(&b.dYb, (size_t)cap * MLP_OUTP) | al(&b.loss, (size_t)cap);
        for (int l = 0; l < 3; l++) bad |= al(&b.Z[l], (size_t)cap * MLP_H);
        for (int l = 0; l < 2; l++) bad |= al(&b.dZ[l], (size_t)cap * MLP_H) | al(&b.dZb[l], (size_t)cap * MLP_H);
        size_t parts = 0;
        for (int l = 0; l < MLP_L; l++) parts += part_floats(cap, l);
        bad |= al(&b.part, parts);
    }
    hipDeviceSynchronize();
    b.cap = bad ? 0 : cap;
    return bad;
}
void mlp_buf_free(MlpBuf &b) {
    void *ps[] = {b.Xb, b.Y, b.dY, b.dYb, b.dZ[0], b.dZ[1], b.dZb[0], b.dZb[1], b.loss, b.Z[0], b.Z[1], b.Z[2],
                  b.Hb[0], b.Hb[1], b.Hb[2], b.part};
    if (b.cap) hipDeviceSynchronize();
    for (void *q : ps)
        if (q) hipFree(q);
    b = MlpBuf();
}
}  // namespace bw

namespace {

int mfail(bw_mlp *m, int code, const std::string &s) {
    if (m) m->err = s;
    return code;
}
#define MCHK(m, x)                                                                                 \
    do {                                                                                           \
        hipError_t e_ = (x);                                                                       \
        if (e_ != hipSuccess) return mfail(m, BW_ERR_HIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
    } while (0)

template <class T>
int malloc0(bw_mlp *m, T **p, size_t n) {
    void *q = nullptr;
    MCHK(m, hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(T)));
    MCHK(m, hipMemsetAsync(q, 0, std::max<size_t>(n, 1) * sizeof(T), m->st));
    MCHK(m, hipStreamSynchronize(m->st));
    m->allocs.push_back(q);
    *p = (T *)q;
    return BW_OK;
}

// The scratch array's device address on the current GPU, looked up once per
// device (the array's host-side name is not a device address).
int scratch_address(bw_mlp *m, unsigned char **out) {
    static std::mutex mu;
    static unsigned char *addr[256] = {};
    int dev = 0;
    MCHK(m, hipGetDevice(&dev));
    if (dev < 0 || dev >= 256) return mfail(m, BW_ERR_HIP, "device index out of range");
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[dev]) {
        void *p = nullptr;
        MCHK(m, hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        addr[dev] = (unsigned char *)p;
    }
    *out = addr[dev];
    return BW_OK;
}

// MlpBuf of n_pad rows carved from the scratch array (forward buffers only)
MlpBuf scratch_buf(unsigned char *base, int n_pad) {
    MlpBuf b;
    b.cap = n_pad;
    size_t o = 0;
    auto take = [&](size_t bytes) {
        unsigned char *p = base + o;
        o += (bytes + 255) / 256 * 256;
        return p;
    };
    b.Xb = (unsigned short *)take((size_t)n_pad * MLP_INP * 2);
    b.Y = (float *)take((size_t)n_pad * MLP_OUTP * 4);
    for (int l = 0; l < 3; l++) b.Hb[l] = (unsigned short *)take((size_t)n_pad * MLP_H * 2);
    return b;
}

unsigned short host_bf16(float f) {
    uint32_t u;
    memcpy(&u, &f, 4);
    if ((u & 0x7f800000u) == 0x7f800000u) return (unsigned short)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

int refresh_bf16(bw_mlp *m) {
    for (int l = 0; l < MLP_L; l++) {
        long long n = (long long)m->K[l] * m->N[l];
        hipLaunchKernelGGL(k_to_bf16, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, m->st, m->W[l], m->Wb[l], n);
    }
    MCHK(m, hipStreamSynchronize(m->st));
    return BW_OK;
}

int ensure_batch(bw_mlp *m, int rows, bool train) {
    if (rows <= m->tb.cap && (m->tb.part || !train)) return BW_OK;
    MCHK(m, hipStreamSynchronize(m->st));
    if (mlp_buf_alloc(m->tb, rows, train)) return mfail(m, BW_ERR_HIP, "hipMalloc (network activations)");
    return BW_OK;
}

// device buffers for n rows of a host call
int ensure_rows(bw_mlp *m, long long n) {
    if (n <= m->xin_rows) return BW_OK;
    MCHK(m, hipStreamSynchronize(m->st));
    for (float **q : {&m->xin, &m->tin, &m->yout}) {
        if (*q) hipFree(*q);
        *q = nullptr;
    }
    m->xin_rows = 0;
    MCHK(m, hipMalloc(&m->xin, sizeof(float) * (size_t)n * MLP_IN));
    MCHK(m, hipMalloc(&m->tin, sizeof(float) * (size_t)n * MLP_T));
    MCHK(m, hipMalloc(&m->yout, sizeof(float) * (size_t)n * MLP_OUT));
    m->xin_rows = n;
    return BW_OK;
}

// the hidden layers over rows [0, n) of device features x (n x 144, raw units;
// idx selects rows, may be null); train: the pre-activations are kept
void forward_hidden(bw_mlp *m, MlpBuf &B, const float *x, const int *idx, int n, int n_pad, bool train, hipStream_t st) {
    long long e = (long long)n_pad * MLP_INP;
    hipLaunchKernelGGL(k_mlp_input, dim3((unsigned)((e + 255) / 256)), dim3(256), 0, st, x, idx, n, n_pad, m->xmean,
                       m->xistd, B.Xb);
    for (int l = 0; l < 3; l++)
        hipLaunchKernelGGL(k_layer, dim3(back_blocks(n_pad, m->N[l])), dim3(256), 0, st, l == 0 ? B.Xb : B.Hb[l - 1], m->Wb[l],
                           m->b[l], n_pad, m->N[l], m->K[l], train ? B.Z[l] : nullptr, B.Hb[l]);
}
// outputs of rows [0, n) in B.Y (n_pad x 32), or in rows (n x 12) if that is not null
void forward(bw_mlp *m, MlpBuf &B, const float *x, const int *idx, int n, int n_pad, hipStream_t st, float *rows = nullptr) {
    forward_hidden(m, B, x, idx, n, n_pad, false, st);
    hipLaunchKernelGGL(k_layer_out, dim3((n_pad + GEMM_B - 1) / GEMM_B), dim3(256), 0, st, B.Hb[2], m->Wb[3], m->b[3], n_pad,
                       B.Y, rows, n);
}

ParamTable param_table(const bw_mlp *m) {
    ParamTable tab{};
    int first = 0, lfirst = 0;
    for (int l = 0; l < MLP_L; l++) {
        const int nw = m->K[l] * m->N[l];
        tab.s[2 * l] = {m->W[l], m->mW[l], m->vW[l], m->Wb[l], nullptr, 0, nw, m->N[l], m->Kl[l], m->Nl[l], first, lfirst};
        first += nw;
        lfirst += m->Kl[l] * m->Nl[l];
        tab.s[2 * l + 1] = {m->b[l], m->mb[l], m->vb[l], nullptr, nullptr, 0, m->N[l], m->N[l], 1, m->Nl[l], first, lfirst};
        first += m->N[l];
        lfirst += m->Nl[l];
    }
    tab.total = first;
    return tab;
}

// losses of rows [0, n) into loss, partial parameter gradients into B.part;
// the returned table holds where they lie.  A weight gradient's batch is split
// into up to WGRAD_SPLITS chunks of whole multiples of 32 rows.
ParamTable loss_backward(bw_mlp *m, MlpBuf &B, const float *x, const float *t, const int *idx, int n, int n_pad, float *loss,
                         hipStream_t st) {
    forward_hidden(m, B, x, idx, n, n_pad, true, st);
    hipLaunchKernelGGL(k_layer_nll, dim3((n_pad + GEMM_B - 1) / GEMM_B), dim3(256), 0, st, B.Hb[2], m->Wb[3], m->b[3], n_pad,
                       t, idx, n, m->tmean, m->tistd, B.dY, B.dYb, loss);
    const int splits = std::max(1, std::min(WGRAD_SPLITS, n_pad / 512));
    const int kc = (n_pad / 32 + splits - 1) / splits * 32, np = (n_pad + kc - 1) / kc;
    const int nb = (n_pad + COLSUM_ROWS - 1) / COLSUM_ROWS;
    ParamTable tab = param_table(m);
    float *part = B.part;
    for (int l = 0; l < MLP_L; l++) {
        tab.s[2 * l].part = part;
        tab.s[2 * l].np = np;
        tab.s[2 * l + 1].part = part + (size_t)WGRAD_SPLITS * m->K[l] * m->N[l];
        tab.s[2 * l + 1].np = nb;
        part += part_floats(B.cap, l);
    }
    const unsigned short *dzb = B.dYb;
    const float *dz = B.dY;
    for (int l = MLP_L - 1; l >= 0; l--) {
        BackArgs a{l == 0 ? B.Xb : B.Hb[l - 1], dzb, m->Wb[l], dz, l == 0 ? nullptr : B.Z[l - 1],
                   (float *)tab.s[2 * l].part, (float *)tab.s[2 * l + 1].part, B.dZ[l & 1], B.dZb[l & 1],
                   n_pad, m->K[l], m->N[l], np, kc};
        const int blocks = (l == 0 ? 0 : back_blocks(n_pad, m->K[l])) + np * back_blocks(m->K[l], m->N[l]) +
                           colsum_blocks(n_pad, m->N[l]);
        hipLaunchKernelGGL(k_layer_back, dim3(blocks), dim3(256), 0, st, a);
        dz = B.dZ[l & 1];
        dzb = B.dZb[l & 1];
    }
    return tab;
}

// parameters in the logical layout: W1 (144x256), b1, W2, b2, W3, b3, W4 (256x12), b4
long long n_params() {
    return (long long)MLP_IN * MLP_H + MLP_H + 2LL * (MLP_H * MLP_H + MLP_H) + (long long)MLP_H * MLP_OUT + MLP_OUT;
}

// parameters (or, from their parts, gradients) to the host
int copy_params(bw_mlp *m, float *out, const ParamTable &tab, bool grads) {
    const dim3 grid((tab.total + 255) / 256), block(256);
    if (grads) hipLaunchKernelGGL(k_pack<true>, grid, block, 0, m->st, tab, m->packed);
    else hipLaunchKernelGGL(k_pack<false>, grid, block, 0, m->st, tab, m->packed);
    MCHK(m, hipMemcpyAsync(out, m->packed, sizeof(float) * n_params(), hipMemcpyDeviceToHost, m->st));
    MCHK(m, hipStreamSynchronize(m->st));
    return BW_OK;
}

}  // namespace

extern "C" {

BW_API int bw_mlp_create(int seed, bw_mlp **out) {
    if (!out) return BW_ERR_ARG;
    bw_mlp *m = new bw_mlp();
    *out = m;
    MCHK(m, hipStreamCreateWithFlags(&m->st, hipStreamNonBlocking));
    int rc;
    if ((rc = scratch_address(m, &m->scratch))) return rc;
    for (int l = 0; l < MLP_L; l++) {
        size_t n = (size_t)m->K[l] * m->N[l];
        if ((rc = malloc0(m, &m->W[l], n)) || (rc = malloc0(m, &m->mW[l], n)) ||
            (rc = malloc0(m, &m->vW[l], n)) || (rc = malloc0(m, &m->Wb[l], n)) ||
            (rc = malloc0(m, &m->b[l], m->N[l])) ||
            (rc = malloc0(m, &m->mb[l], m->N[l])) || (rc = malloc0(m, &m->vb[l], m->N[l])))
            return rc;
    }
    if ((rc = malloc0(m, &m->xmean, MLP_IN)) || (rc = malloc0(m, &m->xistd, MLP_IN)) ||
        (rc = malloc0(m, &m->tmean, MLP_T)) || (rc = malloc0(m, &m->tistd, MLP_T)) ||
        (rc = malloc0(m, &m->packed, (size_t)n_params())))
        return rc;
    // He-uniform initialisation from a splitmix64 stream (logical entries only)
    uint64_t s = (uint64_t)(uint32_t)seed * 0x9E3779B97F4A7C15ull + 0x632BE59BD9B4E019ull;
    auto next = [&]() {
        s += 0x9E3779B97F4A7C15ull;
        uint64_t z = s;
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return (double)((z ^ (z >> 31)) >> 11) * (1.0 / 9007199254740992.0);
    };
    for (int l = 0; l < MLP_L; l++) {
        std::vector<float> w((size_t)m->K[l] * m->N[l], 0.0f);
        double a = std::sqrt(6.0 / m->Kl[l]) * (l == MLP_L - 1 ? 0.1 : 1.0);
        for (int k = 0; k < m->Kl[l]; k++)
            for (int j = 0; j < m->Nl[l]; j++) w[(size_t)k * m->N[l] + j] = (float)((2.0 * next() - 1.0) * a);
        MCHK(m, hipMemcpy(m->W[l], w.data(), sizeof(float) * w.size(), hipMemcpyHostToDevice));
    }
    std::vector<float> one(MLP_IN, 1.0f);
    MCHK(m, hipMemcpy(m->xistd, one.data(), sizeof(float) * MLP_IN, hipMemcpyHostToDevice));
    MCHK(m, hipMemcpy(m->tistd, one.data(), sizeof(float) * MLP_T, hipMemcpyHostToDevice));
    return refresh_bf16(m);
}

BW_API int bw_mlp_destroy(bw_mlp *m) {
    if (!m) return BW_OK;
    if (m->st) hipStreamSynchronize(m->st);
    for (void *q : m->allocs) hipFree(q);
    mlp_buf_free(m->tb);
    for (void *q : {(void *)m->dX, (void *)m->dT, (void *)m->didx, (void *)m->dloss, (void *)m->xin, (void *)m->tin, (void *)m->yout})
        if (q) hipFree(q);
    if (m->ypin) hipHostFree(m->ypin);
    if (m->st) hipStreamDestroy(m->st);
    delete m;
    return BW_OK;
}

BW_API const char *bw_mlp_last_error(bw_mlp *m) { return m ? m->err.c_str() : "no network"; }
BW_API long long bw_mlp_n_params(void) { return n_params(); }

BW_API int bw_mlp_get_params(bw_mlp *m, float *out) {
    if (!m || !out) return BW_ERR_ARG;
    return copy_params(m, out, param_table(m), false);
}

BW_API int bw_mlp_set_params(bw_mlp *m, const float *in) {
    if (!m || !in) return BW_ERR_ARG;
    MCHK(m, hipStreamSynchronize(m->st));
    long long o = 0;
    for (int l = 0; l < MLP_L; l++) {
        std::vector<float> w((size_t)m->K[l] * m->N[l], 0.0f), bb(m->N[l], 0.0f);
        for (int k = 0; k < m->Kl[l]; k++)
            for (int j = 0; j < m->Nl[l]; j++) w[(size_t)k * m->N[l] + j] = in[o++];
        for (int j = 0; j < m->Nl[l]; j++) bb[j] = in[o++];
        MCHK(m, hipMemcpy(m->W[l], w.data(), sizeof(float) * w.size(), hipMemcpyHostToDevice));
        MCHK(m, hipMemcpy(m->b[l], bb.data(), sizeof(float) * bb.size(), hipMemcpyHostToDevice));
    }
    return refresh_bf16(m);
}

// standardisation: x' = (x - x_mean) / x_std (144 each), t' = (t - t_mean) / t_std (6 each)
BW_API int bw_mlp_set_normalisation(bw_mlp *m, const float *x_mean, const float *x_std, const float *t_mean,
                                    const float *t_std) {
    if (!m || !x_mean || !x_std || !t_mean || !t_std) return BW_ERR_ARG;
    std::vector<float> xi(MLP_IN), ti(MLP_T);
    for (int k = 0; k < MLP_IN; k++) xi[k] = x_std[k] > 0 ? 1.0f / x_std[k] : 0.0f;
    for (int k = 0; k < MLP_T; k++) ti[k] = t_std[k] > 0 ? 1.0f / t_std[k] : 0.0f;
    MCHK(m, hipStreamSynchronize(m->st));
    MCHK(m, hipMemcpy(m->xmean, x_mean, sizeof(float) * MLP_IN, hipMemcpyHostToDevice));
    MCHK(m, hipMemcpy(m->xistd, xi.data(), sizeof(float) * MLP_IN, hipMemcpyHostToDevice));
    MCHK(m, hipMemcpy(m->tmean, t_mean, sizeof(float) * MLP_T, hipMemcpyHostToDevice));
    MCHK(m, hipMemcpy(m->tistd, ti.data(), sizeof(float) * MLP_T, hipMemcpyHostToDevice));
    return BW_OK;
}

constexpr int PINNED_ROWS = 1024;
// y (n x 12): standardised mean (6) and log-variance (6) for host features x (n x 144)
BW_API int bw_mlp_forward(bw_mlp *m, const float *x, int n, float *y) {
    if (!m || !x || !y || n < 1) return BW_ERR_ARG;
    int n_pad = (n + 31) / 32 * 32, rc;
    if ((rc = ensure_batch(m, n_pad, false)) || (rc = ensure_rows(m, n))) return rc;
    // (not copies queued on the stream: those of pageable memory take longer,
    // 902 rows 109 us in all against 83; here 75)
    MCHK(m, hipMemcpy(m->xin, x, sizeof(float) * (size_t)n * MLP_IN, hipMemcpyHostToDevice));
    // few rows are written to pinned host memory by the output layer itself (a
    // copy of them would take 10 to 20 us)
    if (n <= PINNED_ROWS && !m->ypin && hipHostMalloc((void **)&m->ypin, sizeof(float) * PINNED_ROWS * MLP_OUT, 0) != hipSuccess) {
        (void)hipGetLastError();
        m->ypin = nullptr;
    }
    const bool pinned = n <= PINNED_ROWS && m->ypin;
    forward(m, m->tb, m->xin, nullptr, n, n_pad, m->st, pinned ? m->ypin : m->yout);
    MCHK(m, hipStreamSynchronize(m->st));
    if (pinned) memcpy(y, m->ypin, sizeof(float) * (size_t)n * MLP_OUT);
    else MCHK(m, hipMemcpy(y, m->yout, sizeof(float) * (size_t)n * MLP_OUT, hipMemcpyDeviceToHost));
    return BW_OK;
}

// bw_mlp_forward on device buffers with no allocation: the activations live
// in the scratch array (n <= NOALLOC_ROWS).  Every buffer it reads is written
// first in the same call, so nothing needs clearing; calls that overlap on one
// GPU share the array and race.
BW_API int bw_mlp_forward_noalloc(bw_mlp *m, const float *x, int n, float *y) {
    if (!m || !x || !y || n < 1) return BW_ERR_ARG;
    if (n > NOALLOC_ROWS)
        return mfail(m, BW_ERR_ARG, "bw_mlp_forward_noalloc: more rows than the scratch array holds (1024)");
    if (!m->scratch) return mfail(m, BW_ERR_STATE, "bw_mlp_forward_noalloc: no scratch address");
    const int n_pad = (n + 31) / 32 * 32;
    MlpBuf B = scratch_buf(m->scratch, n_pad);
    forward(m, B, x, nullptr, n, n_pad, m->st, y);
    MCHK(m, hipGetLastError());
    MCHK(m, hipStreamSynchronize(m->st));
    return BW_OK;
}

// mean loss over n samples and its gradient in the parameter layout
BW_API int bw_mlp_loss_grad(bw_mlp *m, const float *x, const float *t, int n, double *loss, float *grad) {
    if (!m || !x || !t || n < 1) return BW_ERR_ARG;
    int n_pad = (n + 31) / 32 * 32, rc;
    if ((rc = ensure_batch(m, n_pad, true)) || (rc = ensure_rows(m, n))) return rc;
    // (queued, unlike bw_mlp_forward's: two copies and many launches follow, and
    // the waits of plain ones cost more than the slower copies: 20 rows 164
    // against 179 us)
    MCHK(m, hipMemcpyAsync(m->xin, x, sizeof(float) * (size_t)n * MLP_IN, hipMemcpyHostToDevice, m->st));
    MCHK(m, hipMemcpyAsync(m->tin, t, sizeof(float) * (size_t)n * MLP_T, hipMemcpyHostToDevice, m->st));
    const ParamTable tab = loss_backward(m, m->tb, m->xin, m->tin, nullptr, n, n_pad, m->tb.loss, m->st);
    std::vector<float> l(loss ? n : 0);
    if (loss) MCHK(m, hipMemcpyAsync(l.data(), m->tb.loss, sizeof(float) * n, hipMemcpyDeviceToHost, m->st));
    rc = grad ? copy_params(m, grad, tab, true) : BW_OK;
    MCHK(m, hipStreamSynchronize(m->st));  // also after an error: l is a copy's destination
    if (rc) return rc;
    if (loss) {
        double s = 0;
        for (int i = 0; i < n; i++) s += l[i];
        *loss = s / n;
    }
    return BW_OK;
}

// Adam training on n samples (x n x 144 raw features, t n x 6 raw targets):
// epochs over shuffled mini-batches; loss_out[e] = mean loss of epoch e
BW_API int bw_mlp_train(bw_mlp *m, const float *x, const float *t, int n, int epochs, int batch, float lr,
                        int seed, double *loss_out) {
    if (!m || !x || !t || n < 1 || epochs < 1 || batch < 32) return BW_ERR_ARG;
    batch = batch / 32 * 32;
    int rc;
    if ((rc = ensure_batch(m, batch, true))) return rc;
    MCHK(m, hipStreamSynchronize(m->st));
    if (m->dn < n) {
        for (void *q : {(void *)m->dX, (void *)m->dT, (void *)m->didx, (void *)m->dloss})
            if (q) hipFree(q);
        m->dX = m->dT = m->dloss = nullptr;
        m->didx = nullptr;
        m->dn = 0;
        MCHK(m, hipMalloc(&m->dX, sizeof(float) * (size_t)n * MLP_IN));
        MCHK(m, hipMalloc(&m->dT, sizeof(float) * (size_t)n * MLP_T));
        MCHK(m, hipMalloc(&m->didx, sizeof(int) * (size_t)n));
        MCHK(m, hipMalloc(&m->dloss, sizeof(float) * (size_t)n));
        m->dn = n;
    }
    MCHK(m, hipMemcpy(m->dX, x, sizeof(float) * (size_t)n * MLP_IN, hipMemcpyHostToDevice));
    MCHK(m, hipMemcpy(m->dT, t, sizeof(float) * (size_t)n * MLP_T, hipMemcpyHostToDevice));
    std::vector<int> perm(n);
    for (int i = 0; i < n; i++) perm[i] = i;
    uint64_t s = (uint64_t)(uint32_t)seed * 0x9E3779B97F4A7C15ull + 1;
    std::vector<float> l(n);
    for (int e = 0; e < epochs; e++) {
        for (int i = n - 1; i > 0; i--) {  // Fisher-Yates with splitmix64
            s += 0x9E3779B97F4A7C15ull;
            uint64_t z = s;
            z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
            z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
            z ^= z >> 31;
            int j = (int)(z % (uint64_t)(i + 1));
            std::swap(perm[i], perm[j]);
        }
        MCHK(m, hipMemcpy(m->didx, perm.data(), sizeof(int) * (size_t)n, hipMemcpyHostToDevice));
        int done = 0;
        for (int b0 = 0; b0 + batch <= n || b0 == 0; b0 += batch) {
            const int nb = std::min(batch, n - b0);
            const int n_pad = (nb + 31) / 32 * 32;
            const ParamTable tab = loss_backward(m, m->tb, m->dX, m->dT, m->didx + b0, nb, n_pad, m->dloss + b0, m->st);
            m->adam_t++;
            const float b1 = 0.9f, b2 = 0.999f;
            const float c1 = 1.0f - (float)std::pow(b1, (double)m->adam_t), c2 = 1.0f - (float)std::pow(b2, (double)m->adam_t);
            hipLaunchKernelGGL(k_adam, dim3((tab.total + 255) / 256), dim3(256), 0, m->st, tab, lr, b1, b2, c1, c2, 1e-8f);
            done = b0 + nb;
            if (nb < batch) break;
        }
        MCHK(m, hipGetLastError());
        MCHK(m, hipMemcpyAsync(l.data(), m->dloss, sizeof(float) * done, hipMemcpyDeviceToHost, m->st));
        MCHK(m, hipStreamSynchronize(m->st));
        double tot = 0;
        for (int i = 0; i < done; i++) tot += l[i];
        if (loss_out) loss_out[e] = tot / n;
    }
    return BW_OK;
}

}  // extern "C"

namespace bw {
// features (n x 144 raw, device) -> y_out (n x 12): mean (6) and log-variance
// (6) converted back to physical units (mean = t_mean + t_std mu',
// log-variance = s' + 2 log t_std)
__global__ void k_mlp_unscale(const float *__restrict__ y, int n, const float *__restrict__ tmean,
                              const float *__restrict__ tistd, float *__restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    for (int k = 0; k < MLP_T; k++) {
        const float sd = tistd[k] > 0 ? 1.0f / tistd[k] : 0.0f;
        out[(size_t)i * MLP_OUT + k] = tmean[k] + sd * y[(size_t)i * MLP_OUTP + k];
        const float s = fminf(fmaxf(y[(size_t)i * MLP_OUTP + MLP_T + k], -20.0f), 20.0f);
        out[(size_t)i * MLP_OUT + MLP_T + k] = s + 2.0f * logf(fmaxf(sd, 1e-30f));
    }
}

void mlp_forward_device(bw_mlp *m, MlpBuf &B, const float *x, int n, float *y_out, hipStream_t st) {
    const int n_pad = (n + 31) / 32 * 32;
    forward(m, B, x, nullptr, n, n_pad, st);
    hipLaunchKernelGGL(k_mlp_unscale, dim3((n + 255) / 256), dim3(256), 0, st, B.Y, n, m->tmean, m->tistd, y_out);
}
}  // namespace bw
