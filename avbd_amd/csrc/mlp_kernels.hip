// mlp_kernels.hip -- the learned warm start: a per-vertex MLP
// (24 -> 128 -> 128 -> 128 -> 3, SiLU) that predicts the converged step
// displacement from 1-ring features and replaces the inertial initial guess.
//
// Every matrix product, in inference and in training (forward and backward),
// runs on gfx950's BF16 MFMA with FP32 accumulation
// (v_mfma_f32_16x16x32_bf16, 32-deep products): bf16 operands in HBM,
// operand transposition chosen at compile time, and fused epilogues (bias,
// SiLU, SiLU derivative, FP32 / BF16 stores).  Weights keep an FP32 master
// copy updated by Adam; the bf16 copy is refreshed after each update.
//
// MFMA operand layout (16x16x32, 64 lanes, lane l, r = l % 16, g = l / 16):
//   A (16 x 32, rows x k): lane holds A[r][8g .. 8g+7]
//   B (32 x 16, k x cols): lane holds B[8g .. 8g+7][r]
//   D (16 x 16):           lane holds D[4g .. 4g+3][r]
#include <hip/hip_runtime.h>

#include <cstdint>

#include "internal.hpp"
#include "mlp.hpp"

namespace avbd {

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ __bf16 as_bf16(uint16_t u) { return __builtin_bit_cast(__bf16, u); }

__device__ __forceinline__ uint16_t f2bf(float f) {
    // round to nearest even (NaN kept quiet)
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__device__ __forceinline__ float sigmoidf_(float z) { return 1.f / (1.f + __expf(-z)); }

// C[M x N] = A(M x K) B(K x N) with A(m, k) = TA ? a[k * lda + m] : a[m * lda + k]
// and B(k, n) = TB ? b[n * ldb + k] : b[k * ldb + n].  M, N, K multiples of
// 16; a K that is not a multiple of 32 is zero-filled to the next one.
template <bool TA, bool TB, int EPI>
__global__ __launch_bounds__(256) void gemm_bf16_kernel(const uint16_t* __restrict__ a, int lda,
                                                        const uint16_t* __restrict__ b, int ldb,
                                                        float* __restrict__ c32, uint16_t* __restrict__ c16, int ldc,
                                                        const float* __restrict__ bias, const float* __restrict__ aux,
                                                        int ldaux, int M, int N, int K) {
    const int lane = threadIdx.x & 63;
    const int tile = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int tiles_n = N >> 4;
    if (tile >= (M >> 4) * tiles_n) return;   // whole wavefronts leave together
    const int tm = (tile / tiles_n) << 4, tn = (tile % tiles_n) << 4;
    const int r = lane & 15, g = lane >> 4;
    float4_t acc = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < K; k0 += 32) {
        bf16x8_t av, bv;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int k = k0 + 8 * g + j;
            const int m = tm + r, n = tn + r;
            const bool in = k < K;
            av[j] = as_bf16(in ? (TA ? a[(size_t)k * lda + m] : a[(size_t)m * lda + k]) : (uint16_t)0);
            bv[j] = as_bf16(in ? (TB ? b[(size_t)n * ldb + k] : b[(size_t)k * ldb + n]) : (uint16_t)0);
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, acc, 0, 0, 0);
    }
    const int n = tn + r;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int m = tm + 4 * g + j;
        float v = acc[j];
        const size_t o = (size_t)m * ldc + n;
        if constexpr (EPI == MLP_EPI_F32) {
            c32[o] = v;
        } else if constexpr (EPI == MLP_EPI_BIAS_F32) {
            c32[o] = v + bias[n];
        } else if constexpr (EPI == MLP_EPI_BIAS_SILU) {
            const float z = v + bias[n];
            if (c32) c32[o] = z;                       // pre-activation, kept for the backward pass
            c16[o] = f2bf(z * sigmoidf_(z));
        } else if constexpr (EPI == MLP_EPI_SILU_BWD) {
            const float z = aux[(size_t)m * ldaux + n];
            const float s = sigmoidf_(z);
            c16[o] = f2bf(v * s * (1.f + z * (1.f - s)));
        }
    }
}

// Eight consecutive bf16 (16-byte aligned) as an MFMA operand fragment.
__device__ __forceinline__ bf16x8_t ld_frag(const uint16_t* p) {
    return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(p));
}

// The forward products: C[M x N] = A(M x K) B(K x N) with A row-major and
// B(k, n) = b[n * ldb + k] (weights stored out x in), N = 16 NT, K a
// multiple of 32, lda and ldb multiples of 8 (16-byte fragments).  One
// wavefront owns a 16-row strip and all NT output tiles of it, so each A
// fragment is read once (the one-tile-per-wavefront kernel above reads it NT
// times) and the weight fragments, the same for every strip, come from the
// caches.  The k loop and the MFMA sequence per tile are those of
// gemm_bf16_kernel, so the results are identical.
template <int EPI, int NT>
__global__ __launch_bounds__(256) void gemm_rows_kernel(const uint16_t* __restrict__ a, int lda,
                                                        const uint16_t* __restrict__ b, int ldb,
                                                        float* __restrict__ c32, uint16_t* __restrict__ c16, int ldc,
                                                        const float* __restrict__ bias, int M, int K) {
    const int lane = threadIdx.x & 63;
    const int strip = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (strip >= (M >> 4)) return;   // whole wavefronts leave together
    const int tm = strip << 4;
    const int r = lane & 15, g = lane >> 4;
    float4_t acc[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) acc[t] = float4_t{0.f, 0.f, 0.f, 0.f};
    const uint16_t* arow = a + (size_t)(tm + r) * lda + 8 * g;
    for (int k0 = 0; k0 < K; k0 += 32) {
        const bf16x8_t av = ld_frag(arow + k0);
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const bf16x8_t bv = ld_frag(b + (size_t)(t * 16 + r) * ldb + k0 + 8 * g);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, acc[t], 0, 0, 0);
        }
    }
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int n = t * 16 + r;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int m = tm + 4 * g + j;
            const float v = acc[t][j];
            const size_t o = (size_t)m * ldc + n;
            if constexpr (EPI == MLP_EPI_F32) {
                c32[o] = v;
            } else if constexpr (EPI == MLP_EPI_BIAS_F32) {
                c32[o] = v + bias[n];
            } else if constexpr (EPI == MLP_EPI_BIAS_SILU) {
                const float z = v + bias[n];
                if (c32) c32[o] = z;   // pre-activation, kept for the backward pass
                c16[o] = f2bf(z * sigmoidf_(z));
            }
        }
    }
}

// Normalised bf16 features (rows_pad x 32, zero padding) and FP32 targets
// (rows_pad x 3, zero rows) of a raw batch: (value - mean) / std, as the
// in-step features; norm = feature mean, feature std, target mean, target std.
__global__ __launch_bounds__(256) void stage_batch_kernel(const float* __restrict__ feat, const float* __restrict__ tgt,
                                                          const float* __restrict__ norm, int rows, int rows_pad,
                                                          uint16_t* __restrict__ x16, float* __restrict__ t32) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)rows_pad * kMlpInPad) return;
    const int row = (int)(i / kMlpInPad), col = (int)(i % kMlpInPad);
    x16[i] = row < rows && col < kMlpIn ? f2bf((feat[(size_t)row * kMlpIn + col] - norm[col]) / norm[kMlpIn + col])
                                        : (uint16_t)0;
    if (tgt && col < kMlpOut)
        t32[(size_t)row * kMlpOut + col] =
            row < rows ? (tgt[(size_t)row * kMlpOut + col] - norm[2 * kMlpIn + col]) / norm[2 * kMlpIn + kMlpOut + col]
                       : 0.f;
}

// Output-layer loss gradient: dY = 2 (Y - T) / rows for the first `outs`
// columns of the first `rows` rows (zero in the padding), as bf16; the
// block's squared-error sum goes to loss_part[block] (summed in block order
// by grad_reduce_kernel: one add per element on a single loss word
// serialised 12,288 atomics in L2, 15.9 us at 4,096 rows).
__global__ __launch_bounds__(256) void mse_grad_kernel(const float* __restrict__ y, const float* __restrict__ t,
                                                       uint16_t* __restrict__ dy, int rows, int rows_pad, int ld,
                                                       int outs, float* __restrict__ loss_part) {
    __shared__ float red[4];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    float d = 0.f;
    if (i < rows_pad * ld) {
        const int col = i % ld, row = i / ld;
        if (col < outs && row < rows) d = y[i] - t[(size_t)row * outs + col];
        dy[i] = f2bf(2.f * d / (float)rows);
    }
    float s = d * d;
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) loss_part[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// Weight and bias gradients of all four layers over one chunk of rows:
// dW (out x in) = dZ^T (out x rows) H (rows x in), db = dZ^T 1.  The
// contraction runs over thousands of rows into at most 128 x 128 outputs, so
// it is split over the rows (grid.x chunks; grid.y = layer): a block stages 64
// rows of dZ and H at a time in LDS with the row index innermost (rows pairwise,
// 4-byte LDS stores), so that an MFMA fragment (8 consecutive rows) is one
// 16-byte LDS read, and keeps its whole out x in tile in accumulators; the
// bias is one more MFMA against ones.  Each chunk leaves its FP32 partial
// sums in part[chunk][parameter].  One wavefront per 16 x 16 tile over all
// rows, with 2-byte strided loads, had 64 wavefronts in flight and took
// 88 us per layer at 4,096 rows, and the serial column sums of the bias 483 us.
constexpr int kGradRows = 64;              // rows staged at a time
constexpr int kGradLd = kGradRows + 8;     // LDS row length in bf16 (144 B: 16-byte aligned fragments)

template <int OUT, int IN, int MT, int NT>
__device__ __forceinline__ void grad_tile(const uint16_t* __restrict__ dz, const uint16_t* __restrict__ h, int r0,
                                          int r1, int m_base, int n_base, bool bias, uint16_t* sA, uint16_t* sB,
                                          float* __restrict__ gw, float* __restrict__ gb) {
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    float4_t acc[MT][NT], accb[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) {
        accb[i] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    }
    bf16x8_t ones;
#pragma unroll
    for (int j = 0; j < 8; j++) ones[j] = as_bf16((uint16_t)0x3F80u);
    // transposed staging of 64 rows x W columns: a thread reads 8 columns of
    // two neighbouring rows and stores 8 row pairs
    auto stage = [&](const uint16_t* src, int W, uint16_t* dst, int k0) {
        for (int t = threadIdx.x; t < (kGradRows / 2) * (W / 8); t += 256) {
            const int c = (t % (W / 8)) * 8, k = (t / (W / 8)) * 2;
            uint4 a = make_uint4(0, 0, 0, 0), b = a;
            if (k0 + k < r1) a = *reinterpret_cast<const uint4*>(src + (size_t)(k0 + k) * W + c);
            if (k0 + k + 1 < r1) b = *reinterpret_cast<const uint4*>(src + (size_t)(k0 + k + 1) * W + c);
            const uint32_t av[4] = {a.x, a.y, a.z, a.w}, bv[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                *reinterpret_cast<uint32_t*>(dst + (c + 2 * j) * kGradLd + k) = (av[j] & 0xffffu) | (bv[j] << 16);
                *reinterpret_cast<uint32_t*>(dst + (c + 2 * j + 1) * kGradLd + k) = (av[j] >> 16) | (bv[j] & 0xffff0000u);
            }
        }
    };
    for (int k0 = r0; k0 < r1; k0 += kGradRows) {
        __syncthreads();
        stage(dz, OUT, sA, k0);
        stage(h, IN, sB, k0);
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < kGradRows; kk += 32) {
            bf16x8_t av[MT];
#pragma unroll
            for (int i = 0; i < MT; i++) {
                av[i] = ld_frag(sA + (m_base + 16 * i + r) * kGradLd + kk + 8 * g);
                accb[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[i], ones, accb[i], 0, 0, 0);
            }
#pragma unroll
            for (int j = 0; j < NT; j++) {
                const bf16x8_t bv = ld_frag(sB + (n_base + 16 * j + r) * kGradLd + kk + 8 * g);
#pragma unroll
                for (int i = 0; i < MT; i++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[i], bv, acc[i][j], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int m = m_base + 16 * i + 4 * g + q;
#pragma unroll
            for (int j = 0; j < NT; j++) gw[(size_t)m * IN + n_base + 16 * j + r] = acc[i][j][q];
            if (bias && r == 0) gb[m] = accb[i][q];
        }
}

__global__ __launch_bounds__(256) void grad_partial_kernel(MlpGradIn in, int rows, int chunk, int n_params,
                                                           float* __restrict__ part) {
    __shared__ alignas(16) uint16_t sA[kMlpHidden * kGradLd], sB[kMlpHidden * kGradLd];
    const int l = blockIdx.y, w = threadIdx.x >> 6;
    const int r0 = blockIdx.x * chunk, r1 = min(rows, r0 + chunk);
    float* out = part + (size_t)blockIdx.x * n_params + in.off[l];
    if (l == 0)
        grad_tile<kMlpHidden, kMlpInPad, 2, 2>(in.dz[0], in.h[0], r0, r1, 32 * w, 0, true, sA, sB, out,
                                               out + kMlpHidden * kMlpInPad);
    else if (l < kMlpLayers - 1)
        grad_tile<kMlpHidden, kMlpHidden, 2, 8>(in.dz[l], in.h[l], r0, r1, 32 * w, 0, true, sA, sB, out,
                                                out + kMlpHidden * kMlpHidden);
    else
        grad_tile<kMlpOutPad, kMlpHidden, 1, 2>(in.dz[l], in.h[l], r0, r1, 0, 32 * w, w == 0, sA, sB, out,
                                                out + kMlpOutPad * kMlpHidden);
}

// Gradients = the chunks' partial sums added in chunk order (reproducible);
// the last block adds the loss parts in the same way, into grads[n_params].
__global__ __launch_bounds__(256) void grad_reduce_kernel(const float* __restrict__ part, int chunks, int n_params,
                                                          const float* __restrict__ loss_part, int n_loss,
                                                          float* __restrict__ grads) {
    if (blockIdx.x == gridDim.x - 1) {
        __shared__ double red[256];
        double s = 0;
        for (int k = threadIdx.x; k < n_loss; k += 256) s += loss_part[k];
        red[threadIdx.x] = s;
        __syncthreads();
        for (int st = 128; st > 0; st >>= 1) {
            if ((int)threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
            __syncthreads();
        }
        if (threadIdx.x == 0) grads[n_params] = (float)red[0];
        return;
    }
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n_params) return;
    float s = 0.f;
    for (int k = 0; k < chunks; k++) s += part[(size_t)k * n_params + i];
    grads[i] = s;
}

// Adam on FP32 master weights; refreshes the bf16 copy.
__global__ void adam_kernel(float* __restrict__ w, uint16_t* __restrict__ w16, const float* __restrict__ gw,
                            float* __restrict__ m1, float* __restrict__ m2, int n, float lr, float b1, float b2,
                            float eps, float c1, float c2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float g = gw[i];
    const float a = b1 * m1[i] + (1.f - b1) * g;
    const float b = b2 * m2[i] + (1.f - b2) * g * g;
    m1[i] = a;
    m2[i] = b;
    const float v = w[i] - lr * (a / c1) / (sqrtf(b / c2) + eps);
    w[i] = v;
    if (w16) w16[i] = f2bf(v);
}

inline int blocks_for(int n, int b) { return (n + b - 1) / b; }

}  // namespace

void launch_gemm_bf16(hipStream_t s, bool ta, bool tb, int epi, const uint16_t* a, int lda, const uint16_t* b,
                      int ldb, float* c32, uint16_t* c16, int ldc, const float* bias, const float* aux, int ldaux,
                      int M, int N, int K) {
    if (!ta && tb && epi != MLP_EPI_SILU_BWD && (N == 128 || N == 16) && K % 32 == 0 && lda % 8 == 0 &&
        ldb % 8 == 0) {
        const dim3 grid(blocks_for(M / 16, 4)), block(256);
#define AVBD_ROWS(E_, NT_)                                                                                      \
    if (epi == E_ && N == 16 * NT_) {                                                                           \
        hipLaunchKernelGGL((gemm_rows_kernel<E_, NT_>), grid, block, 0, s, a, lda, b, ldb, c32, c16, ldc, bias, \
                           M, K);                                                                               \
        return;                                                                                                 \
    }
        AVBD_ROWS(MLP_EPI_BIAS_SILU, 8)
        AVBD_ROWS(MLP_EPI_BIAS_F32, 8)
        AVBD_ROWS(MLP_EPI_F32, 8)
        AVBD_ROWS(MLP_EPI_BIAS_SILU, 1)
        AVBD_ROWS(MLP_EPI_BIAS_F32, 1)
        AVBD_ROWS(MLP_EPI_F32, 1)
#undef AVBD_ROWS
    }
    const int tiles = (M / 16) * (N / 16);
    const dim3 grid(blocks_for(tiles, 4)), block(256);
#define AVBD_GEMM(TA_, TB_, E_)                                                                                 \
    if (ta == TA_ && tb == TB_ && epi == E_) {                                                                  \
        hipLaunchKernelGGL((gemm_bf16_kernel<TA_, TB_, E_>), grid, block, 0, s, a, lda, b, ldb, c32, c16, ldc,  \
                           bias, aux, ldaux, M, N, K);                                                          \
        return;                                                                                                 \
    }
    // forward: activations (rows x k) times W stored transposed (out x in)
    AVBD_GEMM(false, true, MLP_EPI_BIAS_SILU)
    AVBD_GEMM(false, true, MLP_EPI_BIAS_F32)
    AVBD_GEMM(false, true, MLP_EPI_F32)
    // backward: dH = dZ W (W stored out x in, i.e. B(k=out, n=in) = w[k * in + n])
    AVBD_GEMM(false, false, MLP_EPI_SILU_BWD)
    AVBD_GEMM(false, false, MLP_EPI_F32)
    // weight gradient: dW (out x in) = dZ^T (out x rows) H (rows x in)
    AVBD_GEMM(true, false, MLP_EPI_F32)
#undef AVBD_GEMM
}

void launch_stage_batch(hipStream_t s, const float* feat, const float* tgt, const float* norm, int rows, int rows_pad,
                        uint16_t* x16, float* t32) {
    hipLaunchKernelGGL(stage_batch_kernel, dim3(blocks_for(rows_pad, 256 / kMlpInPad)), dim3(256), 0, s, feat, tgt,
                       norm, rows, rows_pad, x16, t32);
}

int mlp_loss_parts(int rows_pad) { return blocks_for(rows_pad * kMlpOutPad, 256); }

// One 64-row chunk per block fills the chip from about 4,096 rows (64 chunks x
// 4 layers = 256 blocks); beyond that the chunks grow, so that the partial
// sums the reduction reads stay at 64 x 157 KB.
int mlp_grad_chunk_rows(int rows_pad) {
    const int per = (rows_pad + 63) / 64;
    return (per + kGradRows - 1) / kGradRows * kGradRows;
}
int mlp_grad_chunks(int rows_pad) { return blocks_for(rows_pad, mlp_grad_chunk_rows(rows_pad)); }

void launch_mse_grad(hipStream_t s, const float* y, const float* t, uint16_t* dy, int rows, int rows_pad, int ld,
                     int outs, float* loss_part) {
    hipLaunchKernelGGL(mse_grad_kernel, dim3(blocks_for(rows_pad * ld, 256)), dim3(256), 0, s, y, t, dy, rows,
                       rows_pad, ld, outs, loss_part);
}

void launch_grads(hipStream_t s, const MlpGradIn& in, int rows_pad, int n_params, float* part, const float* loss_part,
                  float* grads) {
    const int chunks = mlp_grad_chunks(rows_pad);
    hipLaunchKernelGGL(grad_partial_kernel, dim3(chunks, kMlpLayers), dim3(256), 0, s, in, rows_pad,
                       mlp_grad_chunk_rows(rows_pad), n_params, part);
    hipLaunchKernelGGL(grad_reduce_kernel, dim3(blocks_for(n_params, 256) + 1), dim3(256), 0, s, part, chunks, n_params,
                       loss_part, mlp_loss_parts(rows_pad), grads);
}

void launch_adam(hipStream_t s, float* w, uint16_t* w16, const float* gw, float* m1, float* m2, int n, float lr,
                 float b1, float b2, float eps, int t) {
    const float c1 = 1.f - powf(b1, (float)t), c2 = 1.f - powf(b2, (float)t);
    hipLaunchKernelGGL(adam_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, s, w, w16, gw, m1, m2, n, lr, b1, b2,
                       eps, c1, c2);
}

}  // namespace avbd
