// Kernels of the learned surrogate: a small MLP trained and evaluated with
// BF16 matrix cores and FP32 accumulation.
//
// Every product of a step is small (1024 x 512 x 512 at the largest), so a
// launch is bound by the latency of its loads and of the launch itself, not
// by bandwidth or the matrix cores.  mlp_gemm therefore spends the chip on
// short K chains: a workgroup owns one 32 x 64 (or, where A is read along its
// columns, 64 x 64) block of C and its eight wavefronts split K between them
// (wavefront w takes the 16-deep steps w, w + 8, ...), each with its own
// accumulators, added through LDS in a fixed order at the end.  Operand
// fragments of v_mfma_f32_32x32x16_bf16 are loaded straight from memory, the
// next step's before the current step's products: an operand stored along K
// gives a lane its eight values in one 16-byte load, one stored across K in
// eight 4-byte loads of two neighbouring columns, which feed two products.
// No LDS staging and no barrier in the loop.  All BF16 arrays are padded with
// zeros to multiples of 64 columns, so no load is guarded or unaligned.
// 16 Adam steps of 192-512-512-193 at batch 1024, a parameter read-back and a
// prediction of 256 rows: 25.0 ms -> 1.15 ms (before: one wavefront per 32 x 32
// block over all of K with guarded 2-byte loads, 187 us for a weight gradient;
// one thread per column walking the batch for a bias gradient, 232 us; and a
// host read of the loss in every step).
//
// Lane l supplies A[l % 32][8 (l / 32) + 0..7] and B[8 (l / 32) + 0..7][l % 32]
// of a step; accumulator r holds C[8 (r / 4) + 4 (l / 32) + r % 4][l % 32].
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels_reduce.hpp"

namespace plamd {

typedef __bf16 mlp_bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t mlp_u32x4 __attribute__((ext_vector_type(4)));
typedef float mlp_floatx16 __attribute__((ext_vector_type(16)));

__host__ __device__ inline uint16_t f32_to_bf16(float f) {
    uint32_t u;
    __builtin_memcpy(&u, &f, 4);
    if ((u & 0x7f800000u) == 0x7f800000u) { // inf / nan: keep, quiet the nan
        return static_cast<uint16_t>((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
    }
    u += 0x7fffu + ((u >> 16) & 1u);
    return static_cast<uint16_t>(u >> 16);
}
__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float z) {
    return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

constexpr int kMlpPad = 64;      // columns of every BF16 array are a multiple of this
constexpr int kMlpThreads = 512; // eight wavefronts
constexpr int kMlpWaves = kMlpThreads / 64;

enum MlpEpilogue : int {
    kEpiGrad = 0,     // C = acc (a weight gradient in the parameter layout)
    kEpiGelu = 1,     // Z = acc + bias (FP32), act = GELU(Z) (BF16)
    kEpiGeluGrad = 2, // act = BF16 of acc * GELU'(Z), its column sums to colpart
    kEpiOut = 3,      // C = acc + bias
    kEpiLoss = 4,     // d = acc + bias - target: loss, act = BF16 of dloss/dy, column sums
};

// C[M x N] = op(A) op(B), contraction length K; strides in elements.
struct GemmArgs {
    const uint16_t *A, *B;
    int lda, ldb;
    int M, N, K;
    float *C;          // kEpiGrad, kEpiOut: M x N, stride N
    const float *bias; // kEpiGelu, kEpiOut, kEpiLoss
    float *Z;          // kEpiGelu out, kEpiGeluGrad in, stride ldact
    uint16_t *act;     // kEpiGelu, kEpiGeluGrad, kEpiLoss: padded BF16 output
    int ldact;
    const float *target; // kEpiLoss: M x N
    const float *colw;   // kEpiLoss: loss weights
    double *loss;        // kEpiLoss: one partial per workgroup
    float *colpart;      // kEpiGeluGrad, kEpiLoss: one row of ldact column sums per row block
    int epi;
};

// Two neighbouring columns of eight rows -> the two columns' fragments.
__device__ __forceinline__ void mlp_split(const uint32_t *v, mlp_bf16x8 &even, mlp_bf16x8 &odd) {
    mlp_u32x4 e, o;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        e[q] = __builtin_amdgcn_perm(v[2 * q + 1], v[2 * q], 0x05040100u);
        o[q] = __builtin_amdgcn_perm(v[2 * q + 1], v[2 * q], 0x07060302u);
    }
    even = __builtin_bit_cast(mlp_bf16x8, e);
    odd = __builtin_bit_cast(mlp_bf16x8, o);
}

// Fragments of one 16-deep step: two columns (rows of C for A) per lane of an
// operand stored across K.  GUARD: rows from K on read as zero (the batch
// dimension, whose rows past K hold other data).
template <bool GUARD>
__device__ __forceinline__ void mlp_load_across(const uint16_t *p, int ld, int c0, int k0, int K, int lane,
                                                uint32_t *v) {
    const int k = k0 + 8 * (lane >> 5);
#pragma unroll
    for (int q = 0; q < 8; q++) {
        const int row = GUARD ? min(k + q, K - 1) : k + q;
        const uint32_t w = *reinterpret_cast<const uint32_t *>(p + static_cast<size_t>(row) * ld + c0 + 2 * (lane & 31));
        v[q] = !GUARD || k + q < K ? w : 0U;
    }
}
__device__ __forceinline__ mlp_bf16x8 mlp_load_along(const uint16_t *p, int ld, int row, int k0, int lane) {
    return *reinterpret_cast<const mlp_bf16x8 *>(p + static_cast<size_t>(row) * ld + k0 + 8 * (lane >> 5));
}

// One workgroup's block of C.  TRA: A is stored K x M; TRB: B is stored N x K.
template <bool TRA, bool TRB> __device__ void mlp_gemm(const GemmArgs &g, unsigned block, float *red) {
    constexpr int MT = TRA ? 2 : 1; // 32-row subtiles
    constexpr int ROWS = 32 * MT;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const unsigned nbn = (g.N + 63) / 64;
    const int rb = static_cast<int>(block / nbn);
    const int r0 = rb * ROWS, c0 = static_cast<int>(block % nbn) * 64;
    mlp_floatx16 acc[MT][2] = {};

    uint32_t av[TRA ? 8 : 1], bv[TRB ? 1 : 8];
    mlp_bf16x8 af[MT], bf[2];
    auto load = [&](int k0) {
        if constexpr (TRA) {
            mlp_load_across<true>(g.A, g.lda, r0, k0, g.K, lane, av);
        } else {
            af[0] = mlp_load_along(g.A, g.lda, r0 + (lane & 31), k0, lane);
        }
        if constexpr (TRB) {
            bf[0] = mlp_load_along(g.B, g.ldb, c0 + (lane & 31), k0, lane);
            bf[1] = mlp_load_along(g.B, g.ldb, c0 + 32 + (lane & 31), k0, lane);
        } else {
            mlp_load_across<TRA>(g.B, g.ldb, c0, k0, g.K, lane, bv);
        }
    };
    const int nsteps = (g.K + 15) / 16;
    if (wave < nsteps) {
        load(wave * 16);
    }
    for (int s = wave; s < nsteps; s += kMlpWaves) {
        mlp_bf16x8 a[MT], b[2];
        if constexpr (TRA) {
            mlp_split(av, a[0], a[MT - 1]);
        } else {
            a[0] = af[0];
        }
        if constexpr (TRB) {
            b[0] = bf[0];
            b[1] = bf[1];
        } else {
            mlp_split(bv, b[0], b[1]);
        }
        if (s + kMlpWaves < nsteps) {
            load((s + kMlpWaves) * 16);
        }
#pragma unroll
        for (int i = 0; i < MT; i++) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
            }
        }
    }
    // the wavefronts' sums: 4..7 leave theirs in LDS, 0..3 add theirs, then
    // every thread adds four entries; an operand read across K interleaves
    // its two subtiles' columns (rows of C for A)
    auto at = [&](int i, int j, int r) {
        const int row = 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3), col = lane & 31;
        return (TRA ? 2 * row + i : 32 * i + row) * 64 + (TRB ? 32 * j + col : 2 * col + j);
    };
    float *slot = red + (wave & 3) * ROWS * 64;
    if (wave >= 4) {
#pragma unroll
        for (int i = 0; i < MT; i++) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    slot[at(i, j, r)] = acc[i][j][r];
                }
            }
        }
    }
    __syncthreads();
    if (wave < 4) {
#pragma unroll
        for (int i = 0; i < MT; i++) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    slot[at(i, j, r)] += acc[i][j][r];
                }
            }
        }
    }
    __syncthreads();
    const int cl = tid & 63, col = c0 + cl;
    const bool in = col < g.N;
    const float bias = g.bias && in ? g.bias[col] : 0.0f;
    float csum = 0.0f;
    double lsum = 0;
    for (int rl = tid >> 6; rl < ROWS; rl += kMlpWaves) {
        const int row = r0 + rl;
        const int e = rl * 64 + cl;
        float z = (red[e] + red[ROWS * 64 + e]) + (red[2 * ROWS * 64 + e] + red[3 * ROWS * 64 + e]);
        z += bias;
        if (row >= g.M) {
            continue;
        }
        const size_t o = static_cast<size_t>(row) * g.ldact + col, oc = static_cast<size_t>(row) * g.N + col;
        switch (g.epi) {
        case kEpiGelu:
            // padded columns stay zero: zero weights give NaN where an
            // activation has overflowed, and the next layer reads them
            z = in ? z : 0.0f;
            g.Z[o] = z;
            g.act[o] = f32_to_bf16(gelu(z));
            break;
        case kEpiGeluGrad:
            z = in ? z * gelu_grad(g.Z[o]) : 0.0f;
            csum += z;
            g.act[o] = f32_to_bf16(z);
            break;
        case kEpiLoss:
            if (in) {
                const float d = z - g.target[oc], w = g.colw[col];
                lsum += static_cast<double>(w) * d * d;
                z = 2.0f * w * d / static_cast<float>(g.M);
                csum += z;
            } else {
                z = 0.0f;
            }
            g.act[o] = f32_to_bf16(z);
            break;
        default:
            if (in) {
                g.C[oc] = z;
            }
            break;
        }
    }
    if (g.epi == kEpiGeluGrad || g.epi == kEpiLoss) {
        __syncthreads();
        red[tid] = csum;
        __syncthreads();
        if (tid < 64) {
            float s = 0.0f;
#pragma unroll
            for (int w = 0; w < kMlpWaves; w++) {
                s += red[64 * w + tid];
            }
            g.colpart[static_cast<size_t>(rb) * g.ldact + c0 + tid] = s;
        }
        if (g.epi == kEpiLoss) {
            const double2 t = block_sum2<kMlpThreads>(double2{lsum, 0});
            if (tid == 0) {
                g.loss[block] = t.x;
            }
        }
    }
}

// Forward products (A along K, B across K)
__global__ __launch_bounds__(kMlpThreads) void k_mlp_forward(const GemmArgs g) {
    __shared__ float red[4 * 32 * 64];
    mlp_gemm<false, false>(g, blockIdx.x, red);
}

// Column sums of colpart[nrows x ld]: a bias gradient.
struct ColsumArgs {
    const float *part;
    int nrows, ld, n;
    float *out;
};

// One layer's backward products in one launch: the weight gradient
// (activations^T dz: both operands across the batch), the previous layer's dz
// (dz W^T) and the bias gradient, all of which need only this layer's dz.
// nz = 0 for the first layer, which has no previous one.
__global__ __launch_bounds__(kMlpThreads) void k_mlp_backward(const GemmArgs gw, unsigned nw, const GemmArgs gz,
                                                              unsigned nz, const ColsumArgs cs) {
    __shared__ float red[4 * 64 * 64];
    unsigned b = blockIdx.x;
    if (b < nw) {
        mlp_gemm<true, false>(gw, b, red);
        return;
    }
    b -= nw;
    if (b < nz) {
        mlp_gemm<false, true>(gz, b, red);
        return;
    }
    b -= nz;
    const int col = static_cast<int>(b) * 64 + (threadIdx.x & 63);
    float s = 0.0f;
    if (col < cs.n) {
        for (int r = threadIdx.x >> 6; r < cs.nrows; r += kMlpWaves) {
            s += cs.part[static_cast<size_t>(r) * cs.ld + col];
        }
    }
    red[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x < 64 && col < cs.n) {
        float t = 0.0f;
#pragma unroll
        for (int w = 0; w < kMlpWaves; w++) {
            t += red[64 * w + threadIdx.x];
        }
        cs.out[col] = t;
    }
}

// Where the flat parameter vector's weight matrices lie, and their padded
// BF16 copies.
struct MlpLayout {
    int64_t woff[3], boff[3]; // matrix l is [woff[l], boff[l])
    int cols[3];
    int64_t bf[3]; // offset of the padded copy
    int ld[3];
};

__device__ __forceinline__ void mlp_store_bf16(const MlpLayout &L, int64_t e, float w, uint16_t *wbf) {
#pragma unroll
    for (int l = 0; l < 3; l++) {
        if (e >= L.woff[l] && e < L.boff[l]) {
            const uint32_t i = static_cast<uint32_t>(e - L.woff[l]);
            const uint32_t row = i / static_cast<uint32_t>(L.cols[l]), col = i - row * static_cast<uint32_t>(L.cols[l]);
            wbf[L.bf[l] + static_cast<int64_t>(row) * L.ld[l] + col] = f32_to_bf16(w);
        }
    }
}

// Adam on FP32 master weights, refreshing the BF16 copies.
__global__ __launch_bounds__(256) void k_adam(float *__restrict__ w, uint16_t *__restrict__ wbf, const MlpLayout L,
                                              float *__restrict__ m, float *__restrict__ v,
                                              const float *__restrict__ g, int64_t n, float lr,
                                              float b1, float b2, float eps, float c1, float c2) {
    const int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (e < n) {
        const float gi = g[e];
        const float mi = b1 * m[e] + (1.0f - b1) * gi;
        const float vi = b2 * v[e] + (1.0f - b2) * gi * gi;
        m[e] = mi;
        v[e] = vi;
        const float wi = w[e] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
        w[e] = wi;
        mlp_store_bf16(L, e, wi, wbf);
    }
}

// BF16 copies of the whole parameter vector's matrices
__global__ __launch_bounds__(256) void k_weights_to_bf16(const float *__restrict__ w, uint16_t *__restrict__ wbf,
                                                         const MlpLayout L, int64_t n) {
    const int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (e < n) {
        mlp_store_bf16(L, e, w[e], wbf);
    }
}

// y[rows x ld] = BF16 of x[rows x cols], zeros from column cols on
__global__ __launch_bounds__(256) void k_to_bf16(const float *__restrict__ x, uint16_t *__restrict__ y, int64_t rows,
                                                 int cols, int ld) {
    const int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (e < rows * ld) {
        const int64_t r = e / ld;
        const int c = static_cast<int>(e - r * ld);
        y[e] = c < cols ? f32_to_bf16(x[r * cols + c]) : static_cast<uint16_t>(0);
    }
}

} // namespace plamd
