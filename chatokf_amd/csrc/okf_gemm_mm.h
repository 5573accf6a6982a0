// okf_gemm_mm.h -- tile GEMMs whose weights are converted to fp16 once per
// tile of tokens.
//
// Y[n][m] = sum_k W[m][k] X[n][k] with X in fp16 as Xt[K / 8][N][8]
// (x_to_octets_kernel): the 8 k of one token that one lane of a
// v_mfma_f32_16x16x32_f16 operand takes are 16 contiguous bytes, and 16
// consecutive tokens are 256.
#pragma once
#include "okf_dq16.h"

namespace okf {

// X fp32 [N][K] -> Xt fp16 [K / 8][N][8] (round to nearest even).  A
// workgroup takes 16 tokens x 64 octets: reads of 32 bytes a lane, four lanes
// to 128 contiguous bytes of a token, stores of 256 contiguous bytes an octet.
static __global__ __launch_bounds__(256) void x_to_octets_kernel(const float *__restrict__ X, uint32_t N, uint32_t K8,
                                                                 half8 *__restrict__ Xt) {
    const uint32_t t = threadIdx.x, n = blockIdx.x * 16 + (t & 15);
    const uint32_t o0 = blockIdx.y * 64 + (t >> 4);
    if (n >= N) return;
    const floatx4 *xr = (const floatx4 *)X + (uint64_t)n * K8 * 2;
    floatx4 v[4][2];
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (o0 + 16 * i < K8) {
            v[i][0] = xr[2 * (o0 + 16 * i)];
            v[i][1] = xr[2 * (o0 + 16 * i) + 1];
        }
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (o0 + 16 * i < K8) {
            half8 h;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                h[e] = (_Float16)v[i][0][e];
                h[4 + e] = (_Float16)v[i][1][e];
            }
            Xt[(uint64_t)(o0 + 16 * i) * N + n] = h;
        }
}

// Four consecutive rows m.. of token n.
__device__ __forceinline__ void mm_store4(float *Y, uint32_t M, uint32_t N, uint32_t m, uint32_t n, const floatx4 &c) {
    if (n >= N) return;
    float *dst = Y + (uint64_t)n * M + m;
    if (m + 3 < M && (M & 3) == 0) {
        *(floatx4 *)dst = c;
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (m + e < M) dst[e] = c[e];
    }
}

// ------------------------------------------------------------------------
// Few tokens: a workgroup takes 16 FM rows x 16 FN tokens, and its NW
// wavefronts split K in steps of 128 (wavefront w steps w, w + NW, ... of the
// workgroup's range).  Lane (r = lane % 16, g = lane / 16) converts piece
// 4 s + g of row r of each row tile straight into its MFMA A operands, so no
// weight passes through LDS and no barrier is met before the final sum of
// the wavefronts' tiles (in wavefront order).  The next step's weights and
// activations are in flight while a step computes.
template <int F, int FM, int FN, int NW>
__global__ __launch_bounds__(NW * 64) void gemm_few_kernel(const uint8_t *__restrict__ W, uint64_t row_bytes,
                                                           uint32_t K, uint32_t M, const half8 *__restrict__ Xt,
                                                           uint32_t N, float *__restrict__ Y, uint32_t sper,
                                                           float *__restrict__ part, const u32x4 *__restrict__ tab_g,
                                                           const uint2 *__restrict__ grid,
                                                           const uint8_t *__restrict__ gt) {
    constexpr uint32_t TAB = dq_tab_rows<F>();
    __shared__ uint2 tab[TAB ? TAB : 1];
    __shared__ floatx4 red[NW][FM * FN][64];
    const uint32_t t = threadIdx.x, lane = t & 63, r16 = lane & 15, g = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t m0 = blockIdx.x * 16 * FM, n0 = blockIdx.y * 16 * FN;
    const uint32_t units = K / 32, steps = (units + 3) / 4;
    const uint32_t s0 = blockIdx.z * sper, s1 = min(steps, s0 + sper);
    if constexpr (TAB > 0) {
        for (uint32_t e = t; e < TAB; e += NW * 64) tab[e] = uint2{tab_g[e][0], tab_g[e][1]};
        __syncthreads();
    }
    const uint8_t *row[FM];
#pragma unroll
    for (int i = 0; i < FM; i++) row[i] = W + (uint64_t)min(m0 + 16 * i + r16, M - 1) * row_bytes;
    const half8 *xp[FN];
#pragma unroll
    for (int j = 0; j < FN; j++) xp[j] = Xt + min(n0 + 16 * j + r16, N - 1);

    struct Stage {
        DqRaw<F> w[FM];
        half8 x[FN][4];
    };
    // (past the end of K a lane re-reads the last piece: every load is
    // unconditional, and what it gives is zeroed below)
    auto load = [&](uint32_t s, Stage &st) {
        const uint32_t u = min(4 * s + g, units - 1);
#pragma unroll
        for (int i = 0; i < FM; i++) dq_load<F>(row[i], u, st.w[i]);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint64_t o = (uint64_t)dq_octet<F>(u, k) * N;
#pragma unroll
            for (int j = 0; j < FN; j++) st.x[j][k] = xp[j][o];
        }
    };
    floatx4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) acc[i][j] = floatx4{0, 0, 0, 0};
    auto compute = [&](uint32_t s, Stage &st) {
        const uint32_t u = min(4 * s + g, units - 1);
        const bool past = 4 * s + g >= units;
        if (4 * s + 4 > units) {  // (the last step of a K that is no multiple of 128)
#pragma unroll
            for (int j = 0; j < FN; j++)
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (past) st.x[j][k] = half8{};
        }
#pragma unroll
        for (int i = 0; i < FM; i++) {
            half8 a[4];
            dq_piece<F>(st.w[i], u, a, tab, grid, gt);
            if (4 * s + 4 > units) {
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (past) a[k] = half8{};
            }
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int j = 0; j < FN; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[k], st.x[j][k], acc[i][j], 0, 0, 0);
        }
    };
    Stage st[2];
    uint32_t s = s0 + wave;
    if (s < s1) {
        load(s, st[0]);
        for (; s < s1; s += 2 * NW) {
            load(s + NW, st[1]);
            __builtin_amdgcn_sched_barrier(0);
            compute(s, st[0]);
            __builtin_amdgcn_sched_barrier(0);
            load(s + 2 * NW, st[0]);
            __builtin_amdgcn_sched_barrier(0);
            if (s + NW < s1) compute(s + NW, st[1]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) red[wave][i * FN + j][lane] = acc[i][j];
    __syncthreads();
    float *dst = part ? part + (uint64_t)blockIdx.z * N * M : Y;
    for (uint32_t q = wave; q < FM * FN; q += NW) {
        floatx4 v = red[0][q][lane];
#pragma unroll
        for (int w = 1; w < NW; w++) v += red[w][q][lane];
        mm_store4(dst, M, N, m0 + 16 * (q / FN) + 4 * g, n0 + 16 * (q % FN) + r16, v);
    }
}

// ------------------------------------------------------------------------
// Many tokens: a 512-thread workgroup takes 16 FM rows x 128 FN tokens.  K
// goes in chunks of 256: the workgroup's lanes convert the next chunk of the
// rows' weights into one half of LDS (each weight once per 128 FN tokens)
// while the eight wavefronts, 16 FN tokens each, multiply the current one
// from the other half; the activations come from Xt straight into the MFMA B
// registers, four K steps of 32 ahead.  One barrier a chunk.
//
// LDS half: the 16 bytes of K step kb (of 8), row tile i, octet g (of 4) and
// row r (of 16) are at 1024 (FM kb + i) + 256 g + 16 (r ^ mc_swz(kb, g)), so a
// read is 1 KB of which each lane takes 16 bytes, every bank the same number
// of times (SQ_LDS_BANK_CONFLICT counts one cycle a read, a sixth of the LDS's).  A write instruction's 16 lanes are 8 pieces of two rows, whose
// octets lie in different K steps or octet columns, all at the same place of
// the 256 bytes of all banks but for the exclusive or, which takes the pieces'
// two rows to 16 different places.  (Unswizzled, the writes took a third of the
// kernel, 17408 x 5120 Q4_K, N = 128: 71.5 us, 47 without them; padding between
// the octet columns instead doubled the reads' time.)
constexpr uint32_t MC_NW = 8, MC_BK = 256;
template <int F>
__device__ __forceinline__ uint32_t mc_swz(uint32_t kb, uint32_t g) {
    // (bit 3 from kb alone: the lanes of a read that share banks keep apart)
    if constexpr (F == Q4_K || F == Q5_K) return 4 * (kb >> 1) + 2 * (g >> 1);
    else if constexpr (F == Q6_K) return 8 * (kb >> 2) + 2 * g;
    else return 2 * kb;
}

struct MmTiles {
    uint32_t tiles_m, tiles_n;  // grid: tiles_m tiles_n workgroups (and kz K ranges in z)
    uint32_t cper;              // chunks of a K range
};

template <int F, int FM, int FN>
__global__ __launch_bounds__(64 * MC_NW, 2) void gemm_many_kernel(
    const uint8_t *__restrict__ W, uint64_t row_bytes, uint32_t K, uint32_t M, const half8 *__restrict__ Xt,
    uint32_t N, float *__restrict__ Y, MmTiles mt, float *__restrict__ part, const u32x4 *__restrict__ tab_g,
    const uint2 *__restrict__ grid, const uint8_t *__restrict__ gt) {
    constexpr uint32_t TAB = dq_tab_rows<F>(), KS = 1024 * FM, HALF = 8 * KS;
    constexpr uint32_t PIECES = 16 * FM * 8, T = 64 * MC_NW, NP = (PIECES + T - 1) / T;  // a chunk's pieces, and a lane's
    __shared__ __attribute__((aligned(1024))) uint8_t As[2 * HALF];
    __shared__ uint2 tab[TAB ? TAB : 1];
    const uint32_t t = threadIdx.x, lane = t & 63, r16 = lane & 15, g = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
    // workgroup b -> XCD b % 8: the N tiles of a row block, which read the
    // same weights, go to one XCD (one after the other)
    const uint32_t total = mt.tiles_m * mt.tiles_n, b = blockIdx.x;
    const uint32_t per = total / 8, rest = total % 8, x = b % 8, q = b / 8;
    const uint32_t tile = x * per + min(x, rest) + q;
    const uint32_t m0 = tile / mt.tiles_n * 16 * FM, n0 = tile % mt.tiles_n * 16 * MC_NW * FN + wave * 16 * FN;
    const uint32_t units = K / 32, chunks = (units + 7) / 8;
    const uint32_t c0 = blockIdx.z * mt.cper, c1 = min(chunks, c0 + mt.cper);
    if constexpr (TAB > 0) {
        for (uint32_t e = t; e < TAB; e += T) tab[e] = uint2{tab_g[e][0], tab_g[e][1]};
        __syncthreads();
    }
    // piece p of a lane: row (T p + t) / 8 of the tile, piece t % 8 of the chunk
    const uint32_t pj = t & 7, pr = t >> 3;
    const uint8_t *wrow[NP];
#pragma unroll
    for (uint32_t p = 0; p < NP; p++) wrow[p] = W + (uint64_t)min(m0 + 8 * MC_NW * p + pr, M - 1) * row_bytes;
    auto has = [&](uint32_t p) { return PIECES % T == 0 || p + 1 < NP || T * p + 8 * pr < PIECES; };
    DqRaw<F> raw[NP];
    auto load_w = [&](uint32_t c, uint32_t p) {
        if (has(p)) dq_load<F>(wrow[p], min(8 * c + pj, units - 1), raw[p]);
    };
    auto put_w = [&](uint32_t c, uint32_t p) {
        if (!has(p)) return;
        const uint32_t u = min(8 * c + pj, units - 1), row = 8 * MC_NW * p + pr;
        half8 h[4];
        dq_piece<F>(raw[p], u, h, tab, grid, gt);
        uint8_t *base = As + (c & 1) * HALF + 1024 * (row >> 4);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t o = dq_octet<F>(pj, i);  // octet of the chunk
            *(half8 *)(base + (o >> 2) * KS + 256 * (o & 3) + 16 * ((row & 15) ^ mc_swz<F>(o >> 2, o & 3))) = h[i];
        }
    };
    // activations of K step kb (32 k): octet 4 kb + g of the lane's tokens
    const half8 *xp[FN];
#pragma unroll
    for (int j = 0; j < FN; j++) xp[j] = Xt + (uint64_t)g * N + min(n0 + 16 * j + r16, N - 1);
    constexpr int XD = 4;  // (8 measured the same)
    half8 xb[XD][FN];
    auto load_x = [&](uint32_t kb, half8 *x) {
        const uint64_t o = (uint64_t)min(kb, units - 1) * 4 * N;
#pragma unroll
        for (int j = 0; j < FN; j++) x[j] = xp[j][o];
    };
    floatx4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) acc[i][j] = floatx4{0, 0, 0, 0};
    auto barrier = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

#pragma unroll
    for (uint32_t p = 0; p < NP; p++) load_w(c0, p);
#pragma unroll
    for (int k = 0; k < XD; k++) load_x(8 * c0 + k, xb[k]);
#pragma unroll
    for (uint32_t p = 0; p < NP; p++) {
        put_w(c0, p);
        load_w(c0 + 1, p);
    }
    barrier();
    // Rows i of K step ks are read one (FN > 1) or two steps ahead, into the
    // registers of the step just multiplied, across the chunks as well where
    // the registers allow (CARRY): a chunk's barrier then stands before its
    // last steps, when every wavefront has their rows in registers and the
    // next chunk's in LDS.
    constexpr int PA = FN > 1 ? 1 : 2;
    constexpr bool CARRY = FM * FN < 18;
    half8 a[PA][FM];
    // (computed anew for each step: eight lane offsets kept through the loop
    // cost the registers that the larger tiles do not have)
    auto a_at = [&](uint32_t c, int ks) {
        uint32_t lo = 256 * g + 16 * r16;
        asm volatile("" : "+v"(lo));
        const uint32_t sw = mc_swz<F>(ks, F == Q4_K || F == Q5_K || F == Q6_K ? lo >> 8 : 0);
        return As + (c & 1) * HALF + ks * KS + (lo ^ (16 * sw));
    };
    static_assert(2 * NP <= 8 - PA, "the next chunk is in LDS before the barrier");
    auto read_first = [&](uint32_t c) {
#pragma unroll
        for (int k = 0; k < PA; k++)
#pragma unroll
            for (int i = 0; i < FM; i++) a[k][i] = *(const half8 *)(a_at(c, k) + 1024 * i);
    };
    if (CARRY) read_first(c0);
    for (uint32_t c = c0; c < c1; c++) {
        const uint32_t nks = min(8u, units - 8 * c);
        if (nks == 8) {
            if (!CARRY) read_first(c);
#pragma unroll
            for (int ks = 0; ks < 8; ks++) {
                if (CARRY && ks == 8 - PA) barrier();
                const uint8_t *an = a_at(ks < 8 - PA ? c : c + 1, (ks + PA) % 8);
#pragma unroll
                for (int i = 0; i < FM; i++) {
#pragma unroll
                    for (int j = 0; j < FN; j++)
                        acc[i][j] =
                            __builtin_amdgcn_mfma_f32_16x16x32_f16(a[ks % PA][i], xb[ks % XD][j], acc[i][j], 0, 0, 0);
                    if (CARRY || ks < 8 - PA) a[ks % PA][i] = *(const half8 *)(an + 1024 * i);
                    __builtin_amdgcn_sched_barrier(0);
                }
                load_x(8 * c + ks + XD, xb[ks % XD]);
                // the next chunk's weights, a piece at a time, and the loads
                // of the one after it
#pragma unroll
                for (uint32_t p = 0; p < NP; p++)
                    if (ks == (int)(2 * p) && c + 1 < c1) {
                        put_w(c + 1, p);
                        load_w(c + 2, p);
                    }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (!CARRY) barrier();
        } else {  // the last chunk of a K that is no multiple of 256
            for (uint32_t ks = 0; ks < nks; ks++) {
                half8 xv[FN];
                load_x(8 * c + ks, xv);
#pragma unroll
                for (int i = 0; i < FM; i++) {
                    const half8 av = *(const half8 *)(a_at(c, ks) + 1024 * i);
#pragma unroll
                    for (int j = 0; j < FN; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, xv[j], acc[i][j], 0, 0, 0);
                }
            }
        }
    }
    float *dst = part ? part + (uint64_t)blockIdx.z * N * M : Y;
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) mm_store4(dst, M, N, m0 + 16 * i + 4 * g, n0 + 16 * j + r16, acc[i][j]);
}

}  // namespace okf
