// Load predictor network on gfx950: a 3-layer MLP (ReLU) with BF16 weights and FP32
// accumulation, trained with masked MSE and Adam. Training batches go row by row in three launches;
// larger ones and wide layers through plain LDS-tiled GEMMs (64x64 tiles, 4x4 per thread).
//
// Parameters (flat FP32 master copy, the BF16 copy is what the GEMMs read):
//   W1[n_in x h1] b1[h1] W2[h1 x h2] b2[h2] W3[h2 x n_out] b3[n_out]   (row-major, x @ W)
#include <hip/hip_bf16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "rgkc_internal.h"

namespace rgkc {
namespace {

constexpr int TM = 64, TN = 64, TK = 16;

__device__ __forceinline__ float ld(const float* p, size_t i) { return p[i]; }
__device__ __forceinline__ float ld(const __hip_bfloat16* p, size_t i) { return __bfloat162float(p[i]); }

// C[M x N] (+)= op(A)[M x K] * op(B)[K x N]; A is FP32 activations/gradients, B is FP32 or BF16.
// op(A)(m, kk) = TA ? A[kk*lda + m] : A[m*lda + kk]; op(B)(kk, n) = TB ? B[n*ldb + kk] : B[kk*ldb + n].
// Epilogue: + bias[n] if bias, ReLU if relu; accumulate adds into C.
template <bool TA, bool TB, typename BT>
__global__ __launch_bounds__(256) void k_gemm(int M, int N, int K, const float* __restrict__ A, int lda,
                                              const BT* __restrict__ B, int ldb, float* __restrict__ C, int ldc,
                                              const float* __restrict__ bias, int relu, int accumulate) {
    __shared__ float As[TK][TM + 1];
    __shared__ float Bs[TK][TN + 1];
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
    float acc[4][4] = {};
    for (int k0 = 0; k0 < K; k0 += TK) {
        for (int i = threadIdx.x; i < TM * TK; i += 256) {
            const int mm = i / TK, kk = i % TK;
            const int gm = m0 + mm, gk = k0 + kk;
            float v = 0.f;
            if (gm < M && gk < K) v = TA ? A[(size_t)gk * lda + gm] : A[(size_t)gm * lda + gk];
            As[kk][mm] = v;
        }
        for (int i = threadIdx.x; i < TN * TK; i += 256) {
            const int nn = i % TN, kk = i / TN;
            const int gn = n0 + nn, gk = k0 + kk;
            float v = 0.f;
            if (gn < N && gk < K) v = TB ? ld(B, (size_t)gn * ldb + gk) : ld(B, (size_t)gk * ldb + gn);
            Bs[kk][nn] = v;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < TK; kk++) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; i++) { a[i] = As[kk][ty * 4 + i]; b[i] = Bs[kk][tx * 4 + i]; }
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int gm = m0 + ty * 4 + i;
        if (gm >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int gn = n0 + tx * 4 + j;
            if (gn >= N) continue;
            float v = acc[i][j];
            if (bias) v += bias[gn];
            if (accumulate) v += C[(size_t)gm * ldc + gn];
            if (relu) v = v > 0.f ? v : 0.f;
            C[(size_t)gm * ldc + gn] = v;
        }
    }
}

// out[n] = sum_m G[m, n]
__global__ void k_colsum(int M, int N, const float* __restrict__ G, float* __restrict__ out) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= N) return;
    float s = 0.f;
    for (int m = 0; m < M; m++) s += G[(size_t)m * N + n];
    out[n] = s;
}

// G[i] *= (H[i] > 0)  (ReLU backward on the stored activation)
__global__ void k_relu_bwd(size_t n, const float* __restrict__ H, float* __restrict__ G) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && !(H[i] > 0.f)) G[i] = 0.f;
}

// Masked MSE: loss = sum(mask * (Y - T)^2) / max(1, sum(mask)); dY = 2 mask (Y - T) / max(1, sum mask).
__global__ void k_mse(size_t n, const float* __restrict__ Y, const float* __restrict__ T, const float* __restrict__ mask,
                      float inv_cnt, float* __restrict__ dY, float* __restrict__ loss) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    float l = 0.f;
    if (i < n) {
        const float m = mask ? mask[i] : 1.f;
        const float d = (Y[i] - T[i]) * m;
        dY[i] = 2.f * d * inv_cnt;
        l = d * d * inv_cnt;
    }
    for (int o = 32; o > 0; o >>= 1) l += __shfl_down(l, o, 64);
    if ((threadIdx.x & 63) == 0 && l != 0.f) atomicAdd(loss, l);
}

// Adam on the FP32 master copy, then refresh the BF16 copy.
__global__ void k_adam(size_t n, float* __restrict__ w, __hip_bfloat16* __restrict__ wb, const float* __restrict__ g,
                       float* __restrict__ m1, float* __restrict__ m2, float lr, float b1, float b2, float eps,
                       float c1, float c2, float wd) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i] + wd * w[i];
    const float a = b1 * m1[i] + (1.f - b1) * gi;
    const float b = b2 * m2[i] + (1.f - b2) * gi * gi;
    m1[i] = a;
    m2[i] = b;
    const float mh = a / c1, vh = b / c2;
    const float nw = w[i] - lr * mh / (sqrtf(vh) + eps);
    w[i] = nw;
    wb[i] = __float2bfloat16(nw);
}

__global__ void k_to_bf16(size_t n, const float* __restrict__ w, __hip_bfloat16* __restrict__ wb) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) wb[i] = __float2bfloat16(w[i]);
}

// ---- batches that go row by row (mlp_by_rows): three launches -----------------------------------------
// A training batch is 16 to 64 rows, so the layers are vector-matrix products whose cost is latency: as
// GEMMs of 64 x 64 tiles over the whole K, two workgroups walked layer 1's 2563 inputs in 160 steps
// (0.57 ms of 16 launches for the gradient of 16 rows, n_in 2563, 128 x 128 hidden, 1024 out). Instead:
//   k_rows_in    layer 1's products, split over K: a workgroup takes kper inputs (kKC at a time) x 64
//                outputs of up to 64 rows and leaves partial sums (summed in a fixed order by the next kernel);
//   k_rows_net   one workgroup per row: the rest of the forward pass, the loss and the activations'
//                gradients, row vectors in LDS, weights read once per row (they stay in L2);
//   k_rows_grad  a thread per parameter sums its gradient over the rows.
// All sums in FP32 as before, in shorter chains.
constexpr int kKC = 32;
constexpr int kRowThreads = 1024;

__global__ __launch_bounds__(256) void k_rows_in(int B, int n_in, int h1, int kper, const float* __restrict__ X,
                                                 const __hip_bfloat16* __restrict__ W, float* __restrict__ part) {
    __shared__ float xs[kKC][65];
    __shared__ float ws[kKC][64];
    const int n0 = blockIdx.x * 64, b0 = blockIdx.z * 64, bn = min(64, B - b0);
    const int kb = blockIdx.y * kper, ke = min(kb + kper, n_in);
    const int n = threadIdx.x & 63, r0 = threadIdx.x >> 6;
    float acc[16] = {};
    for (int k0 = kb; k0 < ke; k0 += kKC) {
        const int kn = min(kKC, ke - k0);
        if (k0 > kb) __syncthreads();
        for (int i = threadIdx.x; i < 64 * kKC; i += 256) {
            const int b = i / kKC, kk = i % kKC;
            xs[kk][b] = (b < bn && kk < kn) ? X[(size_t)(b0 + b) * n_in + k0 + kk] : 0.f;
            const int nn = i % 64, kw = i / 64;
            ws[kw][nn] = (n0 + nn < h1 && kw < kn) ? __bfloat162float(W[(size_t)(k0 + kw) * h1 + n0 + nn]) : 0.f;
        }
        __syncthreads();
        for (int kk = 0; kk < kKC; kk++) {
            const float w = ws[kk][n];
#pragma unroll
            for (int i = 0; i < 16; i++)
                if (4 * i < bn) acc[i] = fmaf(xs[kk][r0 + 4 * i], w, acc[i]);
        }
    }
    if (n0 + n >= h1) return;
#pragma unroll
    for (int i = 0; i < 16; i++)
        if (r0 + 4 * i < bn) part[((size_t)blockIdx.y * B + b0 + r0 + 4 * i) * h1 + n0 + n] = acc[i];
}

// out[n] = sum_k f(k, n) for n < N, k < K; all threads call it. With fewer outputs than threads, groups of
// threads share K and their sums are added in group order. `red` holds kRowThreads floats.
template <typename F, typename O>
__device__ __forceinline__ void row_sum(int K, int N, float* red, F f, O out) {
    const int G = N < kRowThreads ? max(1, min(K, kRowThreads / N)) : 1;
    for (int n0 = 0; n0 < N; n0 += kRowThreads) {
        const int nn = min(N - n0, kRowThreads);
        const int n = (int)threadIdx.x % nn, g = (int)threadIdx.x / nn;
        if (g < G) {
            float s = 0.f;
#pragma unroll 8
            for (int k = g; k < K; k += G) s += f(k, n0 + n);
            red[threadIdx.x] = s;
        }
        __syncthreads();
        if ((int)threadIdx.x < nn) {
            float s = red[threadIdx.x];
            for (int q = 1; q < G; q++) s += red[q * nn + (int)threadIdx.x];
            out(n0 + (int)threadIdx.x, s);
        }
        __syncthreads();
    }
}

// out(j, sum_n W[j][n] v[n]) for j < J, a wave per j
template <typename O>
__device__ __forceinline__ void row_dot(int J, int N, const __hip_bfloat16* W, const float* v, O out) {
    for (int j = threadIdx.x >> 6; j < J; j += kRowThreads / 64) {
        float s = 0.f;
#pragma unroll 8
        for (int n = threadIdx.x & 63; n < N; n += 64) s = fmaf(__bfloat162float(W[(size_t)j * N + n]), v[n], s);
        for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
        if ((threadIdx.x & 63) == 0) out(j, s);
    }
    __syncthreads();
}

// T null: forward only. row_loss[b] receives the row's share of the masked MSE.
__global__ __launch_bounds__(kRowThreads) void k_rows_net(MlpDims d, int B, int S, const __hip_bfloat16* __restrict__ W,
                                                          const float* __restrict__ w32, const float* __restrict__ part,
                                                          const float* __restrict__ T, const float* __restrict__ mask,
                                                          float inv_cnt, float* __restrict__ H1, float* __restrict__ H2,
                                                          float* __restrict__ Y, float* __restrict__ dY,
                                                          float* __restrict__ dH1, float* __restrict__ dH2,
                                                          float* __restrict__ row_loss) {
    extern __shared__ float dyn[];
    float *const red = dyn, *const v1 = red + kRowThreads, *const v2 = v1 + d.h1, *const vo = v2 + d.h2;
    const size_t b = blockIdx.x;
    const __hip_bfloat16 *const W2 = W + d.off_W2(), *const W3 = W + d.off_W3();
    const float *const b1 = w32 + d.off_b1(), *const b2 = w32 + d.off_b2(), *const b3 = w32 + d.off_b3();
    row_sum(S, d.h1, red, [&](int s, int n) { return part[((size_t)s * B + b) * d.h1 + n]; },
            [&](int n, float x) {
                x += b1[n];
                v1[n] = x > 0.f ? x : 0.f;
                H1[b * d.h1 + n] = v1[n];
            });
    row_sum(d.h1, d.h2, red, [&](int k, int n) { return v1[k] * __bfloat162float(W2[(size_t)k * d.h2 + n]); },
            [&](int n, float x) {
                x += b2[n];
                v2[n] = x > 0.f ? x : 0.f;
                H2[b * d.h2 + n] = v2[n];
            });
    float l = 0.f;
    row_sum(d.h2, d.n_out, red, [&](int k, int n) { return v2[k] * __bfloat162float(W3[(size_t)k * d.n_out + n]); },
            [&](int n, float x) {
                const size_t i = b * d.n_out + n;
                x += b3[n];
                Y[i] = x;
                if (T) {
                    const float e = (x - T[i]) * (mask ? mask[i] : 1.f);
                    vo[n] = 2.f * e * inv_cnt;
                    dY[i] = vo[n];
                    l += e * e * inv_cnt;
                }
            });
    if (!T) return;
    red[threadIdx.x] = l;
    __syncthreads();
    for (int o = kRowThreads / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) row_loss[b] = red[0];
    row_dot(d.h2, d.n_out, W3, vo, [&](int j, float x) {
        v2[j] = v2[j] > 0.f ? x : 0.f;
        dH2[b * d.h2 + j] = v2[j];
    });
    row_dot(d.h1, d.h2, W2, v2, [&](int j, float x) { dH1[b * d.h1 + j] = v1[j] > 0.f ? x : 0.f; });
}

__global__ __launch_bounds__(256) void k_rows_grad(MlpDims d, int B, const float* __restrict__ X, const float* __restrict__ H1,
                                                   const float* __restrict__ H2, const float* __restrict__ dY,
                                                   const float* __restrict__ dH1, const float* __restrict__ dH2,
                                                   const float* __restrict__ row_loss, float* __restrict__ G,
                                                   float* __restrict__ loss) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i == 0) {
        float l = 0.f;
        for (int b = 0; b < B; b++) l += row_loss[b];
        *loss = l;
    }
    if (i >= d.total()) return;
    // the parameter's layer: inputs A (ones for a bias), output gradients D of width N
    const float *A, *D;
    size_t o;
    int K, N;
    if (i < d.off_W2()) { A = X; D = dH1; o = i; K = d.n_in; N = d.h1; }
    else if (i < d.off_W3()) { A = H1; D = dH2; o = i - d.off_W2(); K = d.h1; N = d.h2; }
    else { A = H2; D = dY; o = i - d.off_W3(); K = d.h2; N = d.n_out; }
    const int kk = (int)(o / N), n = (int)(o % N);
    float s = 0.f;
    if (kk < K) {
#pragma unroll 8
        for (int b = 0; b < B; b++) s = fmaf(A[(size_t)b * K + kk], D[(size_t)b * N + n], s);
    } else {
        for (int b = 0; b < B; b++) s += D[(size_t)b * N + n];
    }
    G[i] = s;
}

template <bool TA, bool TB, typename BT>
hipError_t gemm(int M, int N, int K, const float* A, int lda, const BT* B, int ldb, float* C, int ldc, const float* bias,
                bool relu, bool acc, hipStream_t s) {
    dim3 grid((N + TN - 1) / TN, (M + TM - 1) / TM);
    hipLaunchKernelGGL((k_gemm<TA, TB, BT>), grid, dim3(256), 0, s, M, N, K, A, lda, B, ldb, C, ldc, bias,
                       relu ? 1 : 0, acc ? 1 : 0);
    return hipGetLastError();
}

inline unsigned nblk(size_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

// ---- host-side operations on device buffers (called by the C ABI layer) --------------------
hipError_t mlp_to_bf16(const float* w, void* wb, size_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_to_bf16, dim3(nblk(n)), dim3(256), 0, s, n, w, (__hip_bfloat16*)wb);
    return hipGetLastError();
}

// Batches that go row by row: up to kRowBatch rows whose vectors fit a workgroup's LDS, and
//  - layers 2 and 3 of at most kRowWeights weights, and kRowReads of them over all rows: k_rows_net reads
//    them once per row, the tiles once per 64 rows. Forward, tiles / rows: 2048 x 2048 x 2048 (8.4 M) 0.50 / 0.58 ms at
//    1 row; 1024 x 1024 x 1024 (2.1 M) 1.26 / 0.82 at 512 rows, 1.55 / 1.62 at 1024.
//  - training: as many products of parameters and rows as k_rows_grad sums (kRowProducts), or as many as the tiles'
//    walk over n_in makes up for. A step, tiles / rows: 100 x 1400 x 1400 x 10 1.23 / 0.64 ms at 256 rows, 2.20 / 2.49 at 1024;
//    1000 x 10000 x 100 x 100 1.93 / 0.60 at 16, 4.6 / 9.3 at 1024; 50000 x 512 x 64 x 64 22.4 / 18.1 at 1024.
//  - forward alone: a walk that is worth it. 16 x 16 x 16 x 16 0.055 / 0.071 ms at 1024 rows, 300 x 64 x 64 x 64 0.19 / 0.14;
//    64 x 128 x 128 x 8000 0.068 / 0.104 at 1 row (a row's outputs are made 1024 at a time).
constexpr int kRowBatch = 1024;
constexpr uint64_t kRowWeights = 1u << 22, kRowReads = 1u << 30, kRowProducts = 1u << 31;
static size_t row_lds(const MlpDims& d) { return ((size_t)kRowThreads + d.h1 + d.h2 + d.n_out) * 4; }
bool mlp_by_rows(const MlpDims& d, int B, bool train) {
    const uint64_t w = (uint64_t)d.h1 * d.h2 + (uint64_t)d.h2 * d.n_out, walk = (uint64_t)d.n_in + d.h1 + d.h2;
    if (B > kRowBatch || row_lds(d) > 60 * 1024 || w > kRowWeights || w * B > kRowReads) return false;
    if (train) return d.total() * B <= kRowProducts || d.total() * B <= (uint64_t)d.n_in << 20;
    return walk >= 256 && (uint64_t)d.n_out <= 4 * walk;
}
// Inputs per workgroup of layer 1: kKC, or as many of them as keep the partial sums within kPartFloats (64 MB; a
// row path has at most 14336 * 1024 outputs of layer 1) and the grid within the device's limit.
constexpr uint64_t kPartFloats = 1u << 24, kPartSplits = 1u << 15;
static int row_kper(const MlpDims& d, int B) {
    const uint64_t most = std::max<uint64_t>(1, std::min(kPartSplits, kPartFloats / ((uint64_t)B * d.h1)));
    const uint64_t chunks = ((uint64_t)d.n_in + kKC - 1) / kKC;
    return (int)((chunks + most - 1) / most) * kKC;
}
static int row_splits(const MlpDims& d, int B) { return (int)(((uint64_t)d.n_in + row_kper(d, B) - 1) / row_kper(d, B)); }
size_t mlp_part_floats(const MlpDims& d, int B) { return (size_t)row_splits(d, B) * B * d.h1; }

hipError_t mlp_rows_forward(const MlpDims& d, const void* wb, const float* w32, const float* X, int B, float* part,
                            const float* T, const float* mask, float mask_sum, float* H1, float* H2, float* Y, float* dY,
                            float* dH1, float* dH2, float* row_loss, hipStream_t s) {
    const __hip_bfloat16* W = (const __hip_bfloat16*)wb;
    const int S = row_splits(d, B);
    hipLaunchKernelGGL(k_rows_in, dim3((d.h1 + 63) / 64, S, (B + 63) / 64), dim3(256), 0, s, B, d.n_in, d.h1, row_kper(d, B), X,
                       W + d.off_W1(), part);
    if (hipError_t e = hipGetLastError()) return e;
    hipLaunchKernelGGL(k_rows_net, dim3(B), dim3(kRowThreads), row_lds(d), s, d, B, S, W, w32, (const float*)part, T, mask,
                       1.f / (mask_sum > 1.f ? mask_sum : 1.f), H1, H2, Y, dY, dH1, dH2, row_loss);
    return hipGetLastError();
}

hipError_t mlp_rows_grad(const MlpDims& d, const float* X, int B, const float* H1, const float* H2, const float* dY,
                         const float* dH1, const float* dH2, const float* row_loss, float* G, float* loss, hipStream_t s) {
    hipLaunchKernelGGL(k_rows_grad, dim3(nblk(d.total())), dim3(256), 0, s, d, B, X, H1, H2, dY, dH1, dH2, row_loss, G, loss);
    return hipGetLastError();
}

// Forward: X[B x I] -> H1, H2 (post-ReLU) and Y[B x O].
hipError_t mlp_forward(const MlpDims& d, const void* wb, const float* w32, const float* X, int B, float* H1, float* H2,
                       float* Y, hipStream_t s) {
    const __hip_bfloat16* W = (const __hip_bfloat16*)wb;
    const __hip_bfloat16 *W1 = W + d.off_W1(), *W2 = W + d.off_W2(), *W3 = W + d.off_W3();
    const float *b1 = w32 + d.off_b1(), *b2 = w32 + d.off_b2(), *b3 = w32 + d.off_b3();
    hipError_t e = gemm<false, false>(B, d.h1, d.n_in, X, d.n_in, W1, d.h1, H1, d.h1, b1, true, false, s);
    if (e) return e;
    e = gemm<false, false>(B, d.h2, d.h1, H1, d.h1, W2, d.h2, H2, d.h2, b2, true, false, s);
    if (e) return e;
    return gemm<false, false>(B, d.n_out, d.h2, H2, d.h2, W3, d.n_out, Y, d.n_out, b3, false, false, s);
}

// Backward of masked MSE through the network; G (flat, same layout as the parameters) receives
// the gradients w.r.t. the BF16 weights and FP32 biases. dY/dH1/dH2 are scratch.
hipError_t mlp_backward(const MlpDims& d, const void* wb, const float* X, int B, const float* H1, const float* H2,
                        const float* Y, const float* T, const float* mask, float mask_sum, float* dY, float* dH1,
                        float* dH2, float* G, float* loss, hipStream_t s) {
    const __hip_bfloat16* W = (const __hip_bfloat16*)wb;
    const __hip_bfloat16 *W2 = W + d.off_W2(), *W3 = W + d.off_W3();
    float *gW1 = G + d.off_W1(), *gb1 = G + d.off_b1(), *gW2 = G + d.off_W2(), *gb2 = G + d.off_b2();
    float *gW3 = G + d.off_W3(), *gb3 = G + d.off_b3();
    const size_t nY = (size_t)B * d.n_out;
    hipError_t e = hipMemsetAsync(loss, 0, sizeof(float), s);
    if (e) return e;
    hipLaunchKernelGGL(k_mse, dim3(nblk(nY)), dim3(256), 0, s, nY, Y, T, mask, 1.f / (mask_sum > 1.f ? mask_sum : 1.f),
                       dY, loss);
    // layer 3: gW3 = H2^T dY ; gb3 = colsum dY ; dH2 = dY W3^T (masked by ReLU)
    if ((e = gemm<true, false>(d.h2, d.n_out, B, H2, d.h2, dY, d.n_out, gW3, d.n_out, nullptr, false, false, s))) return e;
    hipLaunchKernelGGL(k_colsum, dim3(nblk(d.n_out)), dim3(256), 0, s, B, d.n_out, dY, gb3);
    if ((e = gemm<false, true>(B, d.h2, d.n_out, dY, d.n_out, W3, d.n_out, dH2, d.h2, nullptr, false, false, s))) return e;
    hipLaunchKernelGGL(k_relu_bwd, dim3(nblk((size_t)B * d.h2)), dim3(256), 0, s, (size_t)B * d.h2, H2, dH2);
    // layer 2
    if ((e = gemm<true, false>(d.h1, d.h2, B, H1, d.h1, dH2, d.h2, gW2, d.h2, nullptr, false, false, s))) return e;
    hipLaunchKernelGGL(k_colsum, dim3(nblk(d.h2)), dim3(256), 0, s, B, d.h2, dH2, gb2);
    if ((e = gemm<false, true>(B, d.h1, d.h2, dH2, d.h2, W2, d.h2, dH1, d.h1, nullptr, false, false, s))) return e;
    hipLaunchKernelGGL(k_relu_bwd, dim3(nblk((size_t)B * d.h1)), dim3(256), 0, s, (size_t)B * d.h1, H1, dH1);
    // layer 1
    if ((e = gemm<true, false>(d.n_in, d.h1, B, X, d.n_in, dH1, d.h1, gW1, d.h1, nullptr, false, false, s))) return e;
    hipLaunchKernelGGL(k_colsum, dim3(nblk(d.h1)), dim3(256), 0, s, B, d.h1, dH1, gb1);
    return hipGetLastError();
}

hipError_t mlp_adam(size_t n, float* w, void* wb, const float* g, float* m1, float* m2, float lr, int step, float wd,
                    hipStream_t s) {
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
    hipLaunchKernelGGL(k_adam, dim3(nblk(n)), dim3(256), 0, s, n, w, (__hip_bfloat16*)wb, g, m1, m2, lr, b1, b2, eps,
                       c1, c2, wd);
    return hipGetLastError();
}

}  // namespace rgkc
