// okf_gemm.h -- tile GEMM on CDNA4 matrix cores (N > 5, e.g. pp512 prefill)
// and the row dequantizer.
//
// Y[n][m] = sum_k W[m][k] X[n][k].  A 256-thread workgroup computes a
// 128 (rows m) x 128 (columns n) tile in K steps of 64: each step decodes the
// W tile to fp32 with the bit-exact unit decoders, rounds it to fp16 into LDS,
// converts the X tile to fp16 into LDS, then the four wavefronts (2 x 2, each
// 64 x 64) run v_mfma_f32_16x16x32_f16 with fp32 accumulation.  This is the
// reference's tile (LLM/metal/Kernels.metal:226-294: W dequantized to half in
// threadgroup memory, X float -> half, fp32 accumulate) laid out for 64-wide
// wavefronts and MFMA fragments.
#pragma once
#include "okf_common.h"
#include "okf_decode.h"

namespace okf {

constexpr int GB_M = 128, GB_N = 128, GB_K = 64, G_LDS_STRIDE = GB_K + 8;

// 32 floats -> 32 halves (round to nearest even) stored at dst (16-byte aligned).
__device__ __forceinline__ void store_half32(_Float16 *dst, const float *v) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        half8 h;
#pragma unroll
        for (int e = 0; e < 8; e++) h[e] = (_Float16)v[i * 8 + e];
        *(half8 *)(dst + i * 8) = h;
    }
}

__device__ __forceinline__ void zero_half32(_Float16 *dst) {
#pragma unroll
    for (int i = 0; i < 4; i++) *(half8 *)(dst + i * 8) = half8{};
}

// K split: workgroup z of the grid's third dimension takes K range
// [z kper, (z + 1) kper) (kper a multiple of GB_K) and, with part, writes
// its tile to part + z N M (Y's layout) for gemm_ksum_kernel to add.
template <int F>
__global__ __launch_bounds__(256) void gemm_mfma_kernel(const uint8_t *__restrict__ W,
                                                        uint64_t row_bytes, uint32_t K, uint32_t M,
                                                        const float *__restrict__ X, uint32_t N,
                                                        float *__restrict__ Y,
                                                        const uint2 *__restrict__ grid_g,
                                                        const uint8_t *__restrict__ gt, uint32_t kper,
                                                        float *__restrict__ part) {
    __shared__ __attribute__((aligned(16))) _Float16 As[GB_M * G_LDS_STRIDE];
    __shared__ __attribute__((aligned(16))) _Float16 Bs[GB_N * G_LDS_STRIDE];
    __shared__ uint2 grid[F == IQ2_XXS ? 256 : 1];
    if constexpr (F == IQ2_XXS) grid[threadIdx.x] = grid_g[threadIdx.x];

    const uint32_t t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const uint32_t wm = wave >> 1, wn = wave & 1;
    const uint32_t n0 = blockIdx.x * GB_N, m0 = blockIdx.y * GB_M;
    const uint32_t lr = t >> 1, lh = t & 1;  // loader: tile row, 32-wide half
    const uint32_t units = K / 32;
    const uint8_t *wrow = W + (uint64_t)min(m0 + lr, M - 1) * row_bytes;
    const float *xrow = X + (uint64_t)min(n0 + lr, N - 1) * K;

    floatx4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = floatx4{0, 0, 0, 0};

    const uint32_t kb = blockIdx.z * kper, ke = min(K, kb + kper);
    for (uint32_t k0 = kb; k0 < ke; k0 += GB_K) {
        __syncthreads();  // previous step's fragments are consumed (and grid loaded)
        const uint32_t u = k0 / 32 + lh;
        _Float16 *ad = As + lr * G_LDS_STRIDE + lh * 32;
        _Float16 *bd = Bs + lr * G_LDS_STRIDE + lh * 32;
        if (u < units) {
            float w[32], x[32];
            decode_unit<F>(wrow, u, w, grid, gt);
            store_half32(ad, w);
            const float4 *xp = (const float4 *)(xrow + u * 32);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                float4 v = xp[i];
                x[4 * i] = v.x;
                x[4 * i + 1] = v.y;
                x[4 * i + 2] = v.z;
                x[4 * i + 3] = v.w;
            }
            store_half32(bd, x);
        } else {
            zero_half32(ad);
            zero_half32(bd);
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < GB_K / 32; kk++) {
            const uint32_t kc = kk * 32 + (lane >> 4) * 8;
            half8 a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; i++)
                a[i] = *(const half8 *)(As + (wm * 64 + i * 16 + (lane & 15)) * G_LDS_STRIDE + kc);
#pragma unroll
            for (int j = 0; j < 4; j++)
                b[j] = *(const half8 *)(Bs + (wn * 64 + j * 16 + (lane & 15)) * G_LDS_STRIDE + kc);
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    }

    // C fragment: lane holds rows 4*(lane>>4) + e of A (weight rows m) for
    // column lane & 15 of B (token n).
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t m = m0 + wm * 64 + i * 16 + 4 * (lane >> 4);
            const uint32_t n = n0 + wn * 64 + j * 16 + (lane & 15);
            if (n >= N) continue;
            float *dst = (part ? part + (uint64_t)blockIdx.z * N * M : Y) + (uint64_t)n * M + m;
            if (m + 3 < M && (M & 3) == 0) {
                *(float4 *)dst = make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (m + e < M) dst[e] = acc[i][j][e];
            }
        }
}

// Y = the sum of the ks K-range partials of gemm_mfma_kernel, in K order
// (deterministic): 4 consecutive values of Y's N M per thread, all ks loads
// issued first in groups of 8.  vec: float4 accesses (the host sets it
// only when N M is a multiple of 4 and Y is 16-byte aligned, so that every
// partial and Y are too); else one value at a time.
static __global__ __launch_bounds__(256) void gemm_ksum_kernel(const float *__restrict__ part, float *__restrict__ Y,
                                                        uint64_t nm, uint32_t ks, uint32_t vec) {
    const uint64_t e = ((uint64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (e >= nm) return;
    if (vec && e + 4 <= nm) {
        float4 v = *(const float4 *)(part + e);
        for (uint32_t c0 = 1; c0 < ks; c0 += 8) {
            float4 w[8];
#pragma unroll
            for (uint32_t c = 0; c < 8; c++)
                if (c0 + c < ks) w[c] = *(const float4 *)(part + (uint64_t)(c0 + c) * nm + e);
#pragma unroll
            for (uint32_t c = 0; c < 8; c++)
                if (c0 + c < ks) {
                    v.x += w[c].x;
                    v.y += w[c].y;
                    v.z += w[c].z;
                    v.w += w[c].w;
                }
        }
        *(float4 *)(Y + e) = v;
    } else {
        for (uint64_t i = e; i < nm && i < e + 4; i++) {
            float v = part[i];
            for (uint32_t c = 1; c < ks; c++) v += part[(uint64_t)c * nm + i];
            Y[i] = v;
        }
    }
}

// One thread per 32-weight unit of a row; bit-exact with the CPU decoders.
template <int F>
__global__ __launch_bounds__(256) void dequant_row_kernel(const uint8_t *__restrict__ row,
                                                          uint32_t units, float *__restrict__ out,
                                                          const uint2 *__restrict__ grid_g,
                                                          const uint8_t *__restrict__ gt) {
    __shared__ uint2 grid[F == IQ2_XXS ? 256 : 1];
    if constexpr (F == IQ2_XXS) {
        grid[threadIdx.x] = grid_g[threadIdx.x];
        __syncthreads();
    }
    const uint32_t u = blockIdx.x * 256 + threadIdx.x;
    if (u >= units) return;
    float w[32];
    decode_unit<F>(row, u, w, grid, gt);
    float4 *o = (float4 *)(out + (uint64_t)u * 32);
#pragma unroll
    for (int i = 0; i < 8; i++) o[i] = make_float4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
}

// Embedding gather (embedBatch, LLM/Base/MetalEnc.swift:1096-1146): row
// ids[n] of W dequantized into out[n][K], one thread per 32-weight unit;
// bit-exact with dequant_row.  An id outside [0, M) is clamped to the
// nearest row, so a bad id cannot read outside the weights.  A workgroup's
// 256 units are 32 KB of consecutive output: they pass through LDS so that
// a store instruction writes 1 KB in order (a thread's own 128 bytes at a time,
// every store touched 64 lines: 512 rows of 5120 Q4_K 6.7 us).  Up to 64 units
// (one row of 2048) are stored as they are: there the trip through LDS and its
// barrier are what shows (one row of 512, IQ3_S 2.0 us direct, 2.2 through LDS).
template <int F>
__global__ __launch_bounds__(256) void embed_batch_kernel(const uint8_t *__restrict__ W,
                                                          uint64_t row_bytes, uint32_t M,
                                                          const int32_t *__restrict__ ids,
                                                          uint32_t units_per_row, uint32_t units,
                                                          float *__restrict__ out,
                                                          const uint2 *__restrict__ grid_g,
                                                          const uint8_t *__restrict__ gt) {
    constexpr uint32_t ST = 36;  // floats a unit takes in LDS (16 lanes' writes hit different banks)
    __shared__ __attribute__((aligned(16))) float ws[256 * ST];
    __shared__ uint2 grid[F == IQ2_XXS ? 256 : 1];
    const uint32_t t = threadIdx.x, g0 = blockIdx.x * 256;
    if constexpr (F == IQ2_XXS) {
        grid[t] = grid_g[t];
        __syncthreads();
    }
    if (g0 + t < units) {
        const uint32_t n = (g0 + t) / units_per_row, u = (g0 + t) % units_per_row;
        const int32_t id = ids[n];
        const uint32_t row = id < 0 ? 0u : min((uint32_t)id, M - 1);
        float w[32];
        decode_unit<F>(W + (uint64_t)row * row_bytes, u, w, grid, gt);
        auto store = [&](float *d) {
#pragma unroll
            for (int i = 0; i < 8; i++)
                ((float4 *)d)[i] = make_float4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
        };
        if (units <= 64) store(out + t * 32);
        else store(ws + t * ST);
    }
    if (units <= 64) return;
    __syncthreads();
    float4 *o = (float4 *)(out + (uint64_t)g0 * 32);
    const uint32_t n4 = min(256u, units - g0) * 8;
#pragma unroll
    for (uint32_t i = 0; i < 8; i++) {
        const uint32_t f = 256 * i + t;
        if (f < n4) o[f] = *(const float4 *)(ws + (f >> 3) * ST + 4 * (f & 7));
    }
}

}  // namespace okf
