// okf_impl.h -- host-side internals shared by the translation units of
// libokf_quant.so: the context, argument checks, scratch management and the
// per-format launchers.  The launchers are templates instantiated once per
// format in okf_fmt_*.hip (so the formats compile in parallel) and declared
// extern here for okf_quant.hip, which holds the C ABI.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <type_traits>
#include <vector>

#include "../../include/okf_quant.h"
#include "okf_common.h"
#include "okf_decode.h"
#include "okf_gemm.h"
#include "okf_gemv.h"
#include "okf_gemv_wide.h"
#include "okf_gemv_sb.h"
#include "okf_gemm_mm.h"
#include "okf_ffn.h"
#include "okf_ffn_mfma.h"

// one matvec y = W x of a launch group (with X2: x = silu(X) * X2)
struct GemvCall {
    const uint8_t *W;
    const float *X;
    float *Y;
    uint32_t M;
    const float *X2 = nullptr;
};

struct okf_ctx {
    int device = -1;
    hipStream_t stream = nullptr;
    uint2 *grid = nullptr;  // 256 IQ2_XXS grid entries in device memory
    uint8_t *grids = nullptr;  // the grids of IQ2_XS, IQ2_S, IQ3_XXS, IQ3_S, IQ1_S / IQ1_M (GT_* offsets)
    okf::u32x4 *tab = nullptr;   // IQ2_XXS fp16 grid (256 x 8 halves) + sign masks (128): MFMA kernel
    okf::u32x4 *tab8 = nullptr;  // IQ2_XXS int8 grid (256) + sign byte masks (128): dot4 kernels
    size_t max_lds = 65536;  // dynamic LDS a workgroup may use
    // matvec tuning (defaults chosen per shape; OKF_GEMV_* environment
    // variables override them for measurements)
    int gemv_s = 0;      // K split across a workgroup's wavefronts (0 = auto)
    int gemv_wide = -1;  // one-workgroup-per-CU matvec: -1 auto, 0 never, 1 where it fits
    int gemv_sb = -1;    // superblock-per-lane matvec: -1 auto, 0 never, 1 where it fits
    int gemv_sb_rw = 0;  // its rows per workgroup (0 = auto)
    int gemv_sb_t = 0;   // its threads per workgroup (0 = auto)
    int gemv_sb_r = 2;   // its rows per lane for IQ2_XXS (2: each x record read serves two rows; or 1)
    int gemm_ks = 0;     // tile GEMM: the many-token kernel with this many K ranges (0 = auto)
    int q4k_mm = 0xFFF;  // 2..4 columns on the matrix cores, bits mm_bit(F) (0: the dot4 kernels)
    int gemm_plan[4] = {0, 0, 0, 0};  // tile GEMM: this kind, fm, fn, K ranges (plan_mm; fm 0: the plan's choice)
    int gemm_split = 1;  // tile GEMM: K split when the grid is small (0 never)
    int gemm_xh = 1;     // tile GEMM of the formats but Q4_K: fp16 X converted once (0: gemm_mfma_kernel on the same
                         // K ranges, for comparison)
    uint32_t cus = 256;  // compute units of the device
    double fault_rate = 0;
    uint64_t fault_state = 0;
    int last_hip = 0;
    _Float16 *xh = nullptr;  // fp16 copy of the GEMM activations (grown on demand)
    size_t xh_bytes = 0;
    // a captured graph holds the buffer's address: when it is replaced the old one is kept
    // in retired until the context is destroyed (grow_buf)
    bool xh_held = false, part_held = false, cnt_held = false;
    std::vector<void *> retired;
    // okf_parallel_begin .. okf_parallel_end: recorded matvecs
    struct Pending {
        int32_t type;
        uint32_t K;
        uint64_t rb;
        GemvCall call;
    };
    bool grouping = false;
    std::vector<Pending> pending;
    float *part = nullptr;   // split-tile partial sums of the Q4_K GEMM, argmax pairs
    size_t part_bytes = 0;
    uint32_t *cnt = nullptr;  // argmax per-row counters (zero between calls)
    size_t cnt_n = 0;
    bool reserved = false;    // okf_ctx_reserve fixed the scratch sizes: no growth
    uint8_t *scratch = nullptr;  // this device's copy of the static scratch array
    uint32_t *ffn_bar = nullptr;  // the one-launch FFN's grid barrier (zeroed at creation)
    uint32_t *ffn_status = nullptr;  // pinned host word: 1 once a launch's barrier gave up (GPUGate verdict)
    int ffn_fused = 1;            // okf_ffn as one launch with a grid barrier: 1 where it fits and is the faster
                                  // form, 2 wherever it fits, 0 never (two launches)
    int ffn_wg = 1;               // its workgroups per CU, at most
    int ffn_coop = 0;             // launched with hipLaunchCooperativeKernel (1) or as a plain grid
    int q2_mfma = 1;              // Q2_0 Bonsai matvecs on the integer matrix cores (q2m_gemv_kernel; 0: off)
    int q2_ks = 1;                // ... down (R <= 8 rows a workgroup) as the K-split tile (0: rows repeated)
    int ffn_mfma = 1;             // the Bonsai shape on the integer matrix cores (ffn_mfma_kernel; 0: off)
    int ffn_nb[4] = {0, 0, 0, 0}; // its kernels' resident workgroups per CU (0: not yet queried)
    int ffn_spin = 0;             // its barrier's poll limit (0: FF_SPIN)
    int ffn_stall = 0;            // its next launches whose barrier must time out (failure tests)
    int ffn_t = 0;                // its exact-fit variant: threads a workgroup (0: the default, 512)
};

namespace okf_impl {

using namespace okf;


inline bool supported(int32_t t) {
    return t == Q8_0 || t == Q4_K || t == IQ2_XXS || t == Q2_0 || t == Q4_0 || t == IQ4_NL || t == Q5_K ||
           t == Q6_K || t == IQ4_XS || grid_fmt(t);
}

inline int hip_fail(okf_ctx *c, hipError_t e) {
    c->last_hip = (int)e;
    return OKF_E_HIP;
}

// splitmix64 -> uniform [0, 1); deterministic per seed.
inline double next_uniform(uint64_t &s) {
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (double)(z >> 11) * (1.0 / 9007199254740992.0);
}

// Shared prologue of every launch call: arguments, fault injection, device.
inline int begin(okf_ctx *c) {
    if (!c) return OKF_E_ARG;
    if (c->fault_rate > 0 && next_uniform(c->fault_state) < c->fault_rate) return OKF_E_INJECTED;
    if (c->device < 0) return OKF_E_NODEV;
    hipError_t e = hipSetDevice(c->device);
    return e == hipSuccess ? OKF_OK : hip_fail(c, e);
}

inline int check_weight(const okf_weight *w, uint64_t *row_bytes) {
    if (!w || !w->base) return OKF_E_ARG;
    if (!supported(w->ggml_type)) return OKF_E_TYPE;
    if (w->K == 0 || w->M == 0 || w->K % block_elems(w->ggml_type)) return OKF_E_SHAPE;
    *row_bytes = (uint64_t)w->K / block_elems(w->ggml_type) * block_bytes(w->ggml_type);
    const uintptr_t a = (uintptr_t)w->base + w->off;
    // Q4_K kernels read 16-byte header/code chunks; others need 2-byte alignment.
    if (w->ggml_type == Q4_K ? (a & 15) : (a & 1)) return OKF_E_SHAPE;
    return OKF_OK;
}

// The one-launch FFN's failure word (written by the kernel, read by the
// host without a copy): OKF_E_TIMEOUT once, and cleared, after a launch whose
// grid barrier gave up (GPUGate.verdict, LLM/Base/MetalGates.swift:130-142).
inline int take_timeout(okf_ctx *c) {
    volatile uint32_t *w = c->ffn_status;
    if (!w || *w == 0) return OKF_OK;
    *w = 0;
    return OKF_E_TIMEOUT;
}

inline bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

// Raises a kernel's dynamic LDS limit once per device (done: one bit per
// device, shared by every context and thread; a repeated call is harmless).
// The limit is the workgroup's LDS less the kernel's static LDS; a failure
// (which leaves the launch at the default limit) is cleared so that it is
// not reported as the launch's error.
inline void set_lds_attr(const okf_ctx *c, const void *fn, std::atomic<uint64_t> &done) {
    const uint64_t bit = 1ull << (c->device & 63);
    if (done.load(std::memory_order_acquire) & bit) return;
    hipFuncAttributes fa{};
    size_t stat = 0;
    if (hipFuncGetAttributes(&fa, fn) == hipSuccess) stat = fa.sharedSizeBytes;
    if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(c->max_lds - stat)) !=
        hipSuccess)
        (void)hipGetLastError();
    done.fetch_or(bit, std::memory_order_acq_rel);
}

inline int finish(okf_ctx *c) {
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? OKF_OK : hip_fail(c, e);
}

// Rows per slot of gemv_kernel: two (each staged activation read serves both)
// where measured faster: IQ2_XXS with 1..5 columns (16.9 -> 16.4 us at one),
// the generic formats with 2..5 (17408 x 5120, N = 4: 15-18 % faster; at one
// column 10-25 % slower), Q4_K and Q2_0 with 5.  (A three-deep ring for the
// Q4_K matvec measured 3-4 % slower than two once the weight loads were issued
// behind the staging's.)
template <int F, int NC>
constexpr int gemv_rows() {
    return ((F == IQ2_XXS && NC >= 1) || (grid_fmt(F) && NC >= 2) ||
            (NC == 5 && F != Q8_0 && F != Q5_K && F != Q6_K && F != IQ4_XS)) ? 2 : 1;
}

// The workgroup of gemv_kernel for 2..5 columns: its wavefronts W and the K
// split S over them (W / S * GV_SLOTS * R rows), by an estimated time in us
// fitted to MI355X at 2048 x 6144 to 17408 x 5120.  A round of workgroups costs
// its staging and latency plus its rows; workgroups that share a CU (LDS, and
// its wavefronts' registers) add their rows; wavefronts that do not divide over
// the four SIMDs, or fewer than eight on a CU, slow the rows down.  Against
// four wavefronts and no split everywhere (us, N = 2 / 3 / 4 / 5):
//   5120 x 17408   Q4_0 34.6 / 48.1 / 60.8 / 47.7 -> 18.0 / 24.6 / 30.5 / 43.9,
//                  Q8_0 40.0 / 51.2 / 62.0 / 73.5 -> 25.2 / 28.7 / 32.9 / 40.0
//   4096 x 14336   IQ3_XXS 24.5 / 31.3 / 40.0 / 43.7 -> 16.4 / 21.3 / 25.4 / 28.9
//   17408 x 5120   Q6_K 26.1 / 45.4 / 54.8 / 62.2 -> 22.0 / 30.1 / 36.2 / 51.9
//   2048 x 6144    IQ4_XS 9.2 / 11.1 / 13.2 / 15.3 -> 7.2 / 8.7 / 10.0 / 11.4
//   2048 x 2048    Q8_0 4.5 / 5.3 / 6.1 / 7.0 -> 4.2 / 4.9 / 5.5 / 6.1
struct GemvPlan {
    uint32_t W, S;
    float us;
};
template <int F, int NC>
GemvPlan plan_gemv(const okf_ctx *c, uint64_t M, uint32_t K) {
    constexpr uint32_t R = gemv_rows<F, NC>(), MAXW = gemv_max_waves<F, NC>(), L = GV_L;
    constexpr uint8_t forms[][2] = {{4, 1}, {8, 1}, {10, 1}, {12, 1}, {4, 2}, {6, 2},
                                    {8, 2}, {10, 2}, {12, 2}, {4, 4}, {8, 4}, {12, 4}};
    const uint32_t steps = (K / unit_weights<F>() + L - 1) / L;
    const size_t xb = (size_t)NC * K / unit_weights<F>() * unit_lds_bytes<F>() + gemv_tab_rows<F>() * 16;
    const float k = K / 14336.0f, stage = 0.5f + k * (2.3f + 2.05f * NC), row = k * (0.17f + 0.13f * NC);
    GemvPlan best{4, 1, 1e30f};
    // Many short rows take four wavefronts and no split: small workgroups, several
    // on a CU (the four-wavefront instance of these formats does with few enough
    // registers for 12 to 24 wavefronts), stage while others compute; Q8_0 N = 2 at
    // 30000 x 2048 14.4 us, with larger ones 17.9; at 20000 x 4096 17.5 against
    // 18.9.  Below that where larger ones measured slower (larger -> four, us): N = 2
    // Q8_0 6144 x 2048 5.84 -> 5.42, Q2_0 4096 x 2048 4.96 -> 4.48, Q4_0 4096 x 1024
    // 4.30 -> 3.96, Q6_K 12288 x 2048 8.16 -> 7.60; N = 5 Q6_K 10240 x 2048 17.0 ->
    // 13.9, Q8_0 4096 x 1024 6.27 -> 5.73, Q2_0 6144 x 2048 8.99 -> 8.41; N = 4 Q2_0
    // 4096 x 2048 6.95 -> 5.97; N = 3 F16 12288 x 2048 12.0 -> 10.3.
    constexpr bool lean = F == Q8_0 || F == Q2_0 || F == Q4_0 || F == IQ4_NL || F == Q6_K;
    const bool shorts = K <= 2048 && M >= 16ull * c->cus &&
                        ((lean && (NC == 2 || (F == Q6_K && NC != 4) || (F != Q2_0 && K <= 1024))) ||
                         (F == Q2_0 && K > 1024 && M <= 32ull * c->cus && (NC < 5 || M >= 20ull * c->cus)) ||
                         ((F == F16 || F == BF16) && NC >= 3 && M >= 40ull * c->cus) ||
                         (F == F32 && K <= 1024 && M >= 40ull * c->cus));
    // (F32 rows that four wavefronts spread evenly: 8192 x 8192 N = 3 58.2 -> 51.3)
    const bool even = F == F32 && K >= 3072 && M % (32ull * c->cus) == 0;
    const bool many = !c->gemv_s && (shorts || even || (K <= 4096 && M > 64ull * c->cus));
    for (const auto &f : forms) {
        const uint32_t W = f[0], S = f[1], rows = W / S * GV_SLOTS * R;
        if (many && (W > 4 || S > 1)) continue;
        if (F == Q6_K && steps < 2 * S) continue;  // (2048 x 2048, N = 3: 5.5 us without a split, 5.9 with)
        if (W > MAXW || (c->gemv_s && S != std::min<uint32_t>(c->gemv_s, 4))) continue;
        const uint32_t fit = (uint32_t)std::min<size_t>(c->max_lds / (xb + 1024), MAXW / W);
        const uint32_t slots = std::max(1u, fit), cus = std::max(1u, c->cus);
        const uint64_t wgs = (M + rows - 1) / rows, full = wgs / ((uint64_t)cus * slots);
        const uint32_t rest = (uint32_t)((wgs - full * cus * slots + cus - 1) / cus);
        auto round = [&](uint32_t n) {  // n workgroups on a CU
            const uint32_t w = n * W, simd = (w + 3) / 4;
            const float busy = simd >= 2 ? 4.0f * simd / w * (0.4f + 0.6f * w / (4.0f * simd)) : 1.4f;
            return stage * (0.5f + 0.5f * n) + n * rows * row * busy * ((steps + S - 1) / S * S) / steps;
        };
        const float us = 2.0f + full * round(slots) + (rest ? round(rest) : 0.0f);
        if (us < best.us) best = {W, S, us};
    }
    return best;
}

template <int F, int NC, int S, bool SILU, int DX = 0, uint32_t MW = gemv_max_waves<F, NC>()>
void launch_gemv_s(okf_ctx *c, const GemvCall *calls, int n, uint64_t rb, uint32_t K,
                   uint32_t cunits, size_t lds, bool pair = false, uint32_t waves = 4) {
    // Q2_0 and Q8_0 at N = 1: a three-deep ring when a wavefront runs three
    // or more steps (the down projection), so that no step waits for a load
    // issued after the first compute; two otherwise (a third buffer would
    // only re-read).  Measured: Q2_0 2048x6144 4.95 -> 4.75 us.
    if constexpr (DX == 0 && NC == 1 && (F == Q2_0 || F == Q8_0)) {
        const uint32_t steps = (K / unit_weights<F>() + GV_L * S - 1) / (GV_L * S);
        if (steps >= 3) return launch_gemv_s<F, NC, S, SILU, 3>(c, calls, n, rb, K, cunits, lds, pair, waves);
    }
    if constexpr (S == 1 && MW > 4)
        if (waves == 4) return launch_gemv_s<F, NC, S, SILU, DX, 4>(c, calls, n, rb, K, cunits, lds, pair, waves);
    constexpr int R = gemv_rows<F, NC>(), D = DX ? DX : 2;
    const void *fn = (const void *)gemv_kernel<F, NC, R, D, S, SILU, MW>;
    static std::atomic<uint64_t> attr{0};  // devices that have the attribute set
    set_lds_attr(c, fn, attr);
    const uint32_t rows_per_wg = (waves / S) * GV_SLOTS * R;
    GemvGroup g{};
    uint32_t total = 0;
    for (int i = 0; i < n; i++) {
        g.W[i] = calls[i].W;
        g.X[i] = calls[i].X;
        g.X2[i] = calls[i].X2;
        g.Y[i] = calls[i].Y;
        g.M[i] = calls[i].M;
        total += (calls[i].M + rows_per_wg - 1) / rows_per_wg;
        g.end[i] = total;
    }
    g.n = (uint32_t)n;
    if (pair) {  // gate and up rows in the same workgroups: half the row slots each
        g.pair = 1;
        total = (calls[0].M + rows_per_wg / 2 - 1) / (rows_per_wg / 2);
    }
    // the tables the compute reads: IQ2_XXS's LDS rows (copied from c->tab),
    // or the grid formats' device-memory grids
    const u32x4 *tabs = itab_rows(F) ? c->tab8 + itab_at(F) : grid_fmt(F) ? (const u32x4 *)(c->grids + gt_off(F)) : c->tab8;
    hipLaunchKernelGGL((gemv_kernel<F, NC, R, D, S, SILU, MW>), dim3(total), dim3(64 * waves), lds, c->stream,
                       g, rb, K, tabs, cunits);
}

template <int F, int NC, uint32_t SP>
void launch_wide_sp(okf_ctx *c, const GemvCall &call, uint64_t rb, uint32_t K, uint32_t G, size_t lds,
                    uint32_t kmax) {
    // weight ring depth: as deep as the registers allow without spills
    constexpr int D = (F == Q4_K || F == Q8_0) ? (NC == 1 ? 3 : 2)
                      : F == Q2_0                ? (NC == 1 ? 6 : 2)
                                                 : (NC <= 2 ? 6 : NC == 3 ? 4 : 3);
    const void *fn = (const void *)gemv_wide_kernel<F, NC, D, SP>;
    static std::atomic<uint64_t> attr{0};  // devices that have the attribute set
    set_lds_attr(c, fn, attr);
    hipLaunchKernelGGL((gemv_wide_kernel<F, NC, D, SP>), dim3(G), dim3(GW_THREADS), lds, c->stream, call.W,
                       rb, K, call.M, call.X, call.Y, c->tab8, kmax);
}

// Where the one-workgroup-per-CU kernel measured faster on MI355X than the
// many-workgroup one (A/B in one process, configuration shapes): IQ2_XXS
// with 2..5 columns (conflict-free tables; 28.2 -> 22.5 us at N = 4),
// Q4_0 / IQ4_NL and long-K Q2_0 with 4..5 columns, and the Q4_K matvec of rows
// past gemv_sb_kernel's 20480 (8192 x 24576: 45.2 -> 24.9 us).
template <int F, int NC>
bool wide_auto(const okf_ctx *c, uint32_t M, uint32_t K) {
    if (M < 8 * c->cus) return F == Q2_0 && NC >= 4 && K >= 4096;
    if (F == IQ2_XXS) return NC >= 2;
    if (F == Q4_0 || F == IQ4_NL) return NC >= 4;
    if (F == Q2_0) return NC >= 4 && K >= 4096;
    if (F == Q4_K) return NC == 1 && K >= 8192;
    return false;
}

// IQ2_XXS with 2..4 columns on the matrix cores (gemv_wide_iq2mm_kernel):
// true when launched.
template <int NC>
bool launch_iq2mm(okf_ctx *c, const GemvCall &call, uint64_t rb, uint32_t K) {
    const uint32_t G = std::min(c->cus, call.M), units = K / 64, P = (units + GV_L - 1) / GV_L;
    const uint64_t nq = ((call.M + G - 1) / G + 3) / 4, lmax = (nq * P + GM_WAVES - 1) / GM_WAVES;
    const uint32_t kmax = (uint32_t)((lmax + P - 1) / P + 1);
    const size_t lds = GM_TAB * 16 + (size_t)P * GV_L * (GM_UNIT + 2) * 16 + (size_t)GM_WAVES * kmax * 4 * NC * 4;
    const uint32_t sp = (units * 32 + GW_THREADS - 1) / GW_THREADS;
    if (lds > c->max_lds || sp > 3 || nq * P * GM_WAVES >= (1ull << 32)) return false;
    constexpr int D = 2;  // weight ring depth (17408 x 5120, N = 4: 1 19.4, 2 19.5, 3 20.2, 4 20.9, 6 21.2, 8 22.9 us)
    auto go = [&](auto spc) {
        constexpr uint32_t SP = decltype(spc)::value;
        const void *fn = (const void *)gemv_wide_iq2mm_kernel<NC, D, SP>;
        static std::atomic<uint64_t> attr{0};  // devices that have the attribute set
        set_lds_attr(c, fn, attr);
        hipLaunchKernelGGL((gemv_wide_iq2mm_kernel<NC, D, SP>), dim3(G), dim3(GW_THREADS), lds, c->stream,
                           call.W, rb, K, call.M, call.X, call.Y, c->tab, kmax);
    };
    if (sp <= 1) go(std::integral_constant<uint32_t, 1>{});
    else if (sp == 2) go(std::integral_constant<uint32_t, 2>{});
    else go(std::integral_constant<uint32_t, 3>{});
    return true;
}

// The formats with a matrix-core 2..4-column kernel, and their bit in
// okf_ctx::q4k_mm.
constexpr int mm_bit(int f) {
    return f == Q4_K ? 0 : f == Q5_K ? 1 : f == IQ4_XS ? 2 : f == Q8_0 ? 3 : f == IQ3_XXS ? 4 : f == IQ3_S ? 5
         : f == IQ2_XS ? 6 : f == IQ2_S ? 7 : f == IQ1_S ? 8 : f == IQ1_M ? 9 : f == Q2_K ? 10 : f == Q3_K ? 11 : -1;
}

// Q4_K, Q5_K, IQ4_XS, Q8_0, the grid formats, Q2_K and Q3_K with 2..4
// columns on the matrix cores (gemv_wide_mm_kernel): true when launched.
template <int F, int NC>
bool launch_widemm(okf_ctx *c, const GemvCall &call, uint64_t rb, uint32_t K) {
    // (measured on MI355X: at M = 2048 the many-workgroup dot4 kernels are
    // faster, e.g. Q8_0 2048 x 2048 N = 2 5.6 against 14.6 us; Q8_0 at N = 2
    // also at 17408 x 5120, 29.6 against 35.4)
    static_assert(mm_bit(F) >= 0, "matrix-core narrow format");
    if (!(c->q4k_mm & (1 << mm_bit(F))) || K % 64 || call.M < 4096 || (F == Q8_0 && NC < 3)) return false;
    constexpr bool MINS = F == Q4_K || F == Q5_K, HSUM = F == Q2_K || F == Q3_K;
    constexpr uint32_t TABR = (F == IQ1_S || F == IQ1_M) ? 512 : itab_rows(F);
    const uint32_t G = std::min(c->cus, call.M), units = K / 64, P = (units + GV_L - 1) / GV_L;
    const uint64_t nq = ((call.M + G - 1) / G + 3) / 4, lmax = (nq * P + GM_WAVES - 1) / GM_WAVES;
    const uint32_t kmax = (uint32_t)((lmax + P - 1) / P + 1);
    const size_t lds = (size_t)TABR * 16 + (size_t)P * GV_L * (GM_UNIT + (MINS ? 4 : HSUM ? 6 : 2)) * 16 +
                       (size_t)GM_WAVES * kmax * 4 * NC * 4;
    const uint32_t sp = (units * 32 + GW_THREADS - 1) / GW_THREADS;
    if (lds > c->max_lds || sp > 3 || nq * P * GM_WAVES >= (1ull << 32)) return false;
    const u32x4 *tab = itab_rows(F) ? c->tab8 + itab_at(F)
                     : TABR ? (const u32x4 *)(c->grids + gt_off(F)) : nullptr;
    constexpr int D = 2;
    auto go = [&](auto spc) {
        constexpr uint32_t SP = decltype(spc)::value;
        const void *fn = (const void *)gemv_wide_mm_kernel<F, NC, D, SP>;
        static std::atomic<uint64_t> attr{0};  // devices that have the attribute set
        set_lds_attr(c, fn, attr);
        hipLaunchKernelGGL((gemv_wide_mm_kernel<F, NC, D, SP>), dim3(G), dim3(GW_THREADS), lds, c->stream,
                           call.W, rb, K, call.M, call.X, call.Y, tab, kmax);
    };
    if (sp <= 1) go(std::integral_constant<uint32_t, 1>{});
    else if (sp == 2) go(std::integral_constant<uint32_t, 2>{});
    else go(std::integral_constant<uint32_t, 3>{});
    return true;
}

// One workgroup per CU (gemv_wide_kernel) for a single matrix: true when
// launched.
template <int F, int NC>
bool launch_gemv_wide(okf_ctx *c, const GemvCall &call, uint64_t rb, uint32_t K) {
    const int mode = c->gemv_wide;
    if (mode == 0 || (mode < 0 && !wide_auto<F, NC>(c, call.M, K))) return false;
    if constexpr (F == IQ2_XXS && NC >= 2 && NC <= 4)  // (mode 2: the dot2 kernel)
        if (mode != 2 && launch_iq2mm<NC>(c, call, rb, K)) return true;
    constexpr uint32_t UW = unit_weights<F>();
    const uint32_t G = std::min(c->cus, call.M), units = K / UW, P = (units + GV_L - 1) / GV_L;
    const uint64_t nmax = (call.M + G - 1) / G, lmax = (nmax * P + GW_SLOTS - 1) / GW_SLOTS;
    const uint32_t kmax = (uint32_t)((lmax + P - 1) / P + 1);
    const uint64_t cunits = (uint64_t)P * GV_L;
    const size_t lds = (F == IQ2_XXS ? GW_TAB * 16 : 0) + (size_t)NC * cunits * unit_lds_bytes<F>() +
                       (size_t)GW_SLOTS * kmax * NC * sizeof(float);
    // one staging round (x slots per thread <= SP), step indices in 32 bits
    const uint32_t nslots = K / 8, sp = (nslots + GW_THREADS - 1) / GW_THREADS;
    if (lds > c->max_lds || sp > (NC == 1 ? 3u : 1u) || nmax * P * GW_SLOTS >= (1ull << 32)) return false;
    if constexpr (NC == 1)
        if (sp > 1) {
            launch_wide_sp<F, NC, 3>(c, call, rb, K, G, lds, kmax);
            return true;
        }
    launch_wide_sp<F, NC, 1>(c, call, rb, K, G, lds, kmax);
    return true;
}

template <int F, int NC, int T, bool SILU, int R = 1, bool PAIR = false>
void launch_sb_t(okf_ctx *c, const GemvGroup &g, uint32_t total, uint64_t rb, uint32_t K, uint32_t RW, size_t lds,
                 uint32_t sr) {
    auto go = [&](auto src) {
        constexpr int SR = decltype(src)::value;
        const void *fn = (const void *)gemv_sb_kernel<F, NC, R, T, SR, SILU, PAIR>;
        static std::atomic<uint64_t> attr{0};  // devices that have the attribute set
        set_lds_attr(c, fn, attr);
        hipLaunchKernelGGL((gemv_sb_kernel<F, NC, R, T, SR, SILU, PAIR>), dim3(total), dim3(T), lds, c->stream, g, rb, K,
                           RW, (const u32x4 *)c->tab8);
    };
    // (one register buffer: a two-deep ring measured slower at every
    // workgroup size tried, 15.5 against 13.6 us at 17408 x 5120)
    switch (sr) {
        case 1: go(std::integral_constant<int, 1>{}); break;
        case 2: go(std::integral_constant<int, 2>{}); break;
        case 3: go(std::integral_constant<int, 3>{}); break;
        default: go(std::integral_constant<int, 5>{}); break;
    }
}

// Where the superblock-per-lane matvec is the faster one, by the superblocks
// (256 weights) of the call.  Measured on MI355X against gemv_kernel (us,
// gemv_kernel -> superblock): Q4_K 2048 x 2048 (16 K superblocks) 3.4 -> 4.0,
// 6144 x 2048 (49 K) 4.4 -> 4.1; Q5_K 2048 x 2048 3.6 -> 4.2, 3000 x 2816 5.5 ->
// 4.7, 17408 x 5120 16.1 -> 13.3, 5120 x 17408 22.8 -> 15.5; Q8_0 6144 x 2048
// 4.8 -> 5.1, 5120 x 5120 8.8 -> 7.8, 17408 x 5120 22.8 -> 18.2; IQ4_XS 6144 x
// 2048 4.8 -> 5.1, 5120 x 5120 8.1 -> 7.7, 5120 x 17408 22.3 -> 16.7; Q4_0 12288 x
// 3584 (172 K) 7.2 -> 7.7, 17408 x 5120 12.4 -> 11.5, 5120 x 17408 19.9 -> 13.5;
// IQ4_NL 17408 x 5120 (348 K) 14.9 -> 15.3, 60000 x 2048 18.7 -> 17.0, 5120 x 17408
// 22.0 -> 17.2; IQ2_XXS 2048 x 2048 4.1 -> 7.6, 12288 x 3584 9.8 -> 11.4, 17408 x 5120
// 14.9 -> 13.9, 60000 x 2048 16.2 -> 17.6, 120000 x 1536 25.0 -> 22.0, 248320 x 1024
// 33.0 -> 26.6, 248320 x 4096 89.5 -> 83.1, 60000 x 512 10.6 -> 8.9.  okf_ffn (gate
// and up paired, and down; H x D; IQ4_XS's gain is down's):
// 6144 x 2048 Q4_K 10.6 -> 10.8, Q5_K 11.6 -> 11.9, Q8_0 12.5 -> 13.1; 7168 x 3584 Q4_K
// 16.4 -> 16.0, Q5_K 20.7 -> 17.7, IQ4_NL 18.3 -> 19.7; 17408 x 5120 Q4_K 37.2 -> 35.8,
// Q5_K 55.6 -> 41.9, IQ4_XS 50.6 -> 44.9, IQ4_NL 55.6 -> 45.3, Q4_0 52.6 -> 35.7, Q8_0
// 78.7 -> 59.7, IQ2_XXS 41.3 -> 41.9.
// From a sweep of K = 512 .. 17408 and 20 K .. 700 K superblocks, weights from HBM
// (gemv_kernel = 1): short rows of whole 1024s, which leave no lane of gemv_kernel
// idle: IQ4_XS 4096 x 6144 1.12, 5400 x 6144 1.14 (2048 x 12250 0.98), Q8_0 4096 x 6144 and
// 3060 x 8192 1.03; paired, rows of both, IQ4_XS 12500 x 7168 1.07, 25000 x 7168
// 1.10 (26680 x 4608 0.92; 34944 x 5120 1.03, but 0.97 where the weights are in the last-level
// cache), Q4_K 17136 x 7168 1.08, 15000 x 8192 1.10 (35000 x 5120 0.95), IQ4_NL
// 25000 x 7168 1.06.  Long rows with one to one and a half 32-row workgroups a CU, whose
// second round is mostly empty: Q8_0 10000 x 10240 1.05, 9803 x 14336 1.15; paired IQ4_XS 8320 x
// 9216 1.12, 10240 x 17408 1.06 (Q4_K, Q5_K, Q4_0 0.7 to 1.05).
template <int F>
bool sb_auto(uint64_t rows, uint32_t K, bool pair, uint32_t cus) {
    const uint32_t nsb = K / 256;
    const uint64_t n = rows * nsb;  // (paired: of both matrices)
    const bool lng = K > 8192, tail = lng && rows > 32ull * cus && rows <= 48ull * cus, whole = K % 1024 == 0;
    if (pair) {
        switch (F) {
            case Q4_K:
            case IQ4_XS: return n >= 190000 && (lng ? F == Q4_K || !tail : K <= 6144 || !whole);
            case Q5_K: return n >= 190000;
            // (the pair's rows leave a tenth of the 256 lanes idle)
            case IQ4_NL: return n >= 380000 && (lng || !whole || (256 / nsb & ~1u) * nsb >= 230);
            default: return n >= 380000;
        }
    }
    switch (F) {
        case Q4_K: return lng || n >= 30000;
        case Q5_K: return n >= 30000;
        case IQ2_XXS: return (n >= 100000 && K >= 5120) || rows >= 120000 || (K <= 512 && rows >= 50000);
        case Q4_0: return n >= (lng ? 96000u : 300000u);
        case IQ4_NL: return n >= (lng ? 96000u : 400000u);
        case IQ4_XS: return n >= (lng || K <= 5120 || !whole ? 96000u : 140000u);
        default: return n >= (lng || K <= 5120 || !whole ? 96000u : 110000u) && !tail;  // Q8_0
    }
}

// Superblock-per-lane matvec (gemv_sb_kernel): true when launched.  Short
// rows (<= 32 superblocks): T = 256 lanes and RW = T / nsb rows, one
// superblock per lane (IQ2_XXS: two rows per lane, RW = 2 T / nsb).  Long
// rows: T = 512 and RW = M / CUs (one workgroup per CU, each lane a few
// superblocks), so that the per-workgroup staging of x is shared by more
// rows.
template <int F, int NC, bool SILU>
bool launch_gemv_sb(okf_ctx *c, const GemvCall *calls, int n, uint64_t rb, uint32_t K, bool pair = false) {
    if constexpr (!sb_fmt<F>() || NC > 1 || (SILU && F != Q4_K && F != IQ2_XXS)) {
        return false;
    } else {
        const uint32_t nsb = K / 256;
        if (c->gemv_sb == 0 || K % 256) return false;
        uint32_t M = 0;
        for (int i = 0; i < n; i++) M += calls[i].M;
        if (c->gemv_sb < 0 && !sb_auto<F>(M, K, pair, c->cus)) return false;
        const bool lng = nsb > 32;
        if (F == IQ2_XXS && (lng || pair)) return false;  // (long or paired rows: gemv_kernel is no slower)
        uint32_t T = c->gemv_sb_t ? (uint32_t)c->gemv_sb_t : lng ? 512 : 256;
        if (T != 256 && T != 512) T = 256;
        // staging rounds: at most five (K <= 20480), which the registers hold; with
        // nine, 73 to 175 registers a lane spilled (us, gemv_kernel or
        // gemv_wide_kernel -> nine rounds, 8192 x 28672: Q8_0 77 -> 253, Q5_K 65 ->
        // 154, Q4_0 62 -> 110, IQ4_NL 68 -> 101, IQ4_XS 57 -> 93, Q4_K 51 -> 109)
        const uint32_t sr = (K / 8 + T - 1) / T;
        if (sr > 5) return false;
        uint32_t RW = c->gemv_sb_rw ? (uint32_t)c->gemv_sb_rw
                      : lng       ? std::min(32u, std::max(4u, (M + c->cus - 1) / c->cus))
                                  : std::max(1u, T / nsb) * (F == IQ2_XXS && c->gemv_sb_r == 2 ? 2 : 1);
        // (short rows: down, so that the items fill no second round: 21 rows of 12
        // superblocks are 252 items, 22 are 264 on 256 lanes: gate and up, 9564 x 3072 together 229 K
        // superblocks, against gemv_kernel IQ4_XS 1.23 of its time with 22 rows, 0.96 with 20,
        // Q4_K 1.09 and 0.88)
        if (pair) RW = lng || c->gemv_sb_rw ? RW + (RW & 1) : RW & ~1u;
        const size_t lds = (size_t)sb_tab_rows<F>() * 16 + ((size_t)NC * nsb * SB_CHUNKS * 16) +
                           (size_t)RW * nsb * NC * sizeof(float) + (pair ? RW * sizeof(float) : 0);
        if (lds > c->max_lds) return false;
        GemvGroup g{};
        uint32_t total = 0;
        for (int i = 0; i < n; i++) {
            g.W[i] = calls[i].W;
            g.X[i] = calls[i].X;
            g.X2[i] = calls[i].X2;
            g.Y[i] = calls[i].Y;
            g.M[i] = calls[i].M;
            total += (calls[i].M + RW - 1) / RW;
            g.end[i] = total;
        }
        g.n = (uint32_t)n;
        if (pair) total = (calls[0].M + RW / 2 - 1) / (RW / 2);
        const bool two = F == IQ2_XXS && c->gemv_sb_r == 2 && T == 256 && RW % 2 == 0;
        if constexpr (!SILU)
            if (pair) {
                if constexpr (F != IQ2_XXS) {
                    if (T == 256) launch_sb_t<F, NC, 256, false, 1, true>(c, g, total, rb, K, RW, lds, sr);
                    else launch_sb_t<F, NC, 512, false, 1, true>(c, g, total, rb, K, RW, lds, sr);
                }
                return true;
            }
        if (two) launch_sb_t<F, NC, 256, SILU, F == IQ2_XXS ? 2 : 1>(c, g, total, rb, K, RW, lds, sr);
        else if (T == 256) launch_sb_t<F, NC, 256, SILU>(c, g, total, rb, K, RW, lds, sr);
        else launch_sb_t<F, NC, 512, SILU>(c, g, total, rb, K, RW, lds, sr);
        return true;
    }
}

// Launch geometry: for one column 256-thread workgroups of four wavefronts,
// each four row slots of 16 lanes; with fewer than ~3072 wavefronts' worth of
// rows, K is split two ways across the wavefronts of a workgroup (more, shorter
// wavefronts; a four-way split loses to the extra activation staging it
// needs).  For more columns as plan_gemv says.
template <int F, int NC, bool SILU = false>
void launch_gemv_nc(okf_ctx *c, const GemvCall *calls, int n, uint64_t rb, uint32_t K) {
    if (launch_gemv_sb<F, NC, SILU>(c, calls, n, rb, K)) return;
    if constexpr (mm_bit(F) >= 0 && !SILU && NC >= 2 && NC <= 4)
        if (n == 1 && launch_widemm<F, NC>(c, calls[0], rb, K)) return;
    // (Q4_K and Q8_0 units are too large for a deep ring at N > 1; the
    // formats added after the measurements take the many-workgroup kernel)
    if constexpr (!SILU && !((F == Q4_K || F == Q8_0) && NC > 1) && F != Q5_K && F != Q6_K && F != IQ4_XS &&
                  !grid_fmt(F))  // (IQ3_XXS included: the wide kernel has no tables for it)
        if (n == 1 && launch_gemv_wide<F, NC>(c, calls[0], rb, K)) return;
    constexpr uint32_t UW = unit_weights<F>();
    const size_t tab = gemv_tab_rows<F>() * 16;
    const uint32_t units = K / UW;
    // stage all of x when it fits, else in chunks of 64-unit groups (per
    // 32 weights: three 32-byte digit planes and a float4 of group data)
    const size_t per_unit = (size_t)NC * unit_lds_bytes<F>();
    uint32_t rows = 0, waves = 4, S = 1;
    for (int i = 0; i < n; i++) rows += calls[i].M;
    if constexpr (NC > 1) {
        const GemvPlan p = plan_gemv<F, NC>(c, rows, K);
        if constexpr (NC >= 4 && gemv_max_waves<F, NC>() == 4) {
            // two launches of fewer columns, on more wavefronts (Q4_K
            // 5120 x 17408, N = 4: 63.7 -> 40.6 us)
            if (n == 1 && plan_gemv<F, 2>(c, rows, K).us + plan_gemv<F, NC - 2>(c, rows, K).us < p.us) {
                GemvCall call = calls[0];
                launch_gemv_nc<F, 2, SILU>(c, &call, 1, rb, K);
                call.X += 2 * (uint64_t)K;
                call.Y += 2 * (uint64_t)call.M;
                return launch_gemv_nc<F, NC - 2, SILU>(c, &call, 1, rb, K);
            }
        }
        waves = p.W;
        S = p.S;
    }
    const size_t red = waves * GV_SLOTS * NC * 4 * sizeof(float);
    uint32_t cunits = (units + 63) / 64 * 64;
    const size_t budget = c->max_lds - tab - red;
    if (cunits * per_unit > budget) cunits = (uint32_t)(budget / per_unit) / 64 * 64;
    const size_t lds = tab + cunits * per_unit + red;
    const uint32_t waves1 = (rows + GV_SLOTS - 1) / GV_SLOTS;  // wavefronts without a split
    if (NC == 1) S = c->gemv_s ? (uint32_t)c->gemv_s : waves1 < 3072 ? 2 : 1;
    if (S >= 4) launch_gemv_s<F, NC, 4, SILU>(c, calls, n, rb, K, cunits, lds, false, waves);
    else if (S == 2) launch_gemv_s<F, NC, 2, SILU>(c, calls, n, rb, K, cunits, lds, false, waves);
    else launch_gemv_s<F, NC, 1, SILU>(c, calls, n, rb, K, cunits, lds, false, waves);
}

// Q2_0 matvecs of the Bonsai shapes on the integer matrix cores
// (q2m_gemv_kernel, okf_ffn_mfma.h): K = 2048 (gate / up, alone or paired
// with the SiLU) or 6144 (down, with or without the SiLU formed in the
// staging), one workgroup per CU; true when launched.
inline bool launch_q2m(okf_ctx *c, const GemvCall &g0, const GemvCall *g1, uint64_t rb, uint32_t K) {
    if (!c->q2_mfma || !c->cus || (K != 2048 && K != 6144) || (g1 && (K != 2048 || g1->M != g0.M))) return false;
    const uint32_t G = c->cus, R = (g0.M + G - 1) / G, nt = ((g1 ? 2 : 1) * R + 15) / 16;
    // Eight wavefronts (with sixteen, each a half of the K blocks, gate / up
    // took 4.89 against 4.09 us and down 4.33 against 4.25; with four, gate /
    // up 4.40 against 4.14); twelve for the K-split down, so that every
    // thread stages one slot of its 6144 values (3.67 against 3.76 us).
    constexpr uint32_t nw = 8, nwk = 12;
    const bool ks = K == 6144 && !g1 && nt == 1 && R <= 8 && c->q2_ks;
    const size_t lds = q2m_lds_bytes(K, ks ? nwk : nw);
    if (lds > c->max_lds || nt > 3) return false;
    const Q2mArgs a{g0.W, g1 ? g1->W : nullptr, rb, K, g0.M, g0.X, g0.X2, g0.Y, g1 ? g1->Y : nullptr};
    const void *fn = nullptr;
    if (K == 2048 && g1 && !g0.X2) fn = nt == 3 ? (const void *)q2m_gemv_kernel<2, 3, true, false, nw> : nullptr;
    else if (K == 2048 && !g0.X2) fn = nt == 2 ? (const void *)q2m_gemv_kernel<2, 2, false, false, nw> : nullptr;
    else if (ks)
        fn = g0.X2 ? (const void *)q2m_gemv_kernel<4, 1, false, true, nwk, true>
                   : (const void *)q2m_gemv_kernel<4, 1, false, false, nwk, true>;
    else if (K == 6144 && !g1 && nt == 1)
        fn = g0.X2 ? (const void *)q2m_gemv_kernel<6, 1, false, true, nw>
                   : (const void *)q2m_gemv_kernel<6, 1, false, false, nw>;
    if (!fn) return false;
    void *args[] = {(void *)&a};
    if (hipLaunchKernel(fn, dim3(G), dim3((ks ? nwk : nw) * 64), args, lds, c->stream) == hipSuccess) return true;
    (void)hipGetLastError();  // (the caller's fallback launch is the call's result)
    return false;
}

// okf_ffn's two launches both on q2m_gemv_kernel (gate / up K 2048, down K
// 6144): then they are faster than the one launch with its grid barrier
// (8.6 against 9.5 us a step), so okf_ffn takes them unless told otherwise.
inline bool q2m_ffn_fits(const okf_ctx *c, uint32_t ka, uint32_t ma, uint32_t mb) {
    if (!c->q2_mfma || !c->cus || ka != 2048 || ma != 6144) return false;
    const uint32_t G = c->cus, ra = (ma + G - 1) / G, rb = (mb + G - 1) / G;
    return (2 * ra + 15) / 16 == 3 && (rb + 15) / 16 == 1 && q2m_lds_bytes(6144, 12) <= c->max_lds;
}

template <int F>
void launch_gemv(okf_ctx *c, const GemvCall *calls, int n, uint64_t rb, uint32_t K, uint32_t N) {
    if constexpr (F == Q2_0)
        if (n == 1 && N == 1 && launch_q2m(c, calls[0], nullptr, rb, K)) return;
    if (calls[0].X2) {  // SiLU-gated activations: one column
        launch_gemv_nc<F, 1, true>(c, calls, n, rb, K);
        return;
    }
    switch (N) {
    case 1: launch_gemv_nc<F, 1>(c, calls, n, rb, K); break;
    case 2: launch_gemv_nc<F, 2>(c, calls, n, rb, K); break;
    case 3: launch_gemv_nc<F, 3>(c, calls, n, rb, K); break;
    case 4: launch_gemv_nc<F, 4>(c, calls, n, rb, K); break;
    default: launch_gemv_nc<F, 5>(c, calls, n, rb, K); break;
    }
}

// The FFN's gate and up (one format, same shape, shared x) in one grid
// whose workgroups each take the same rows of both: gate <- silu(gate x) *
// (up x), up <- up x.  The down projection then reads one activation vector
// with no SiLU in its staging.
template <int F>
void launch_gemv_pair(okf_ctx *c, const GemvCall *calls, uint64_t rb, uint32_t K) {
    if constexpr (F == Q2_0)
        if (launch_q2m(c, calls[0], &calls[1], rb, K)) return;
    if (launch_gemv_sb<F, 1, false>(c, calls, 2, rb, K, true)) return;
    constexpr uint32_t UW = unit_weights<F>();
    const size_t tab = gemv_tab_rows<F>() * 16;
    const uint32_t units = K / UW;
    const size_t per_unit = unit_lds_bytes<F>();
    const size_t red = 4 * GV_SLOTS * 4 * sizeof(float);
    uint32_t cunits = (units + 63) / 64 * 64;
    const size_t budget = c->max_lds - tab - red;
    if (cunits * per_unit > budget) cunits = (uint32_t)(budget / per_unit) / 64 * 64;
    launch_gemv_s<F, 1, 1, false>(c, calls, 2, rb, K, cunits, tab + cunits * per_unit + red, true);
}

// The FFN block of Q2_0 gate / up / down in one launch (grid barrier)
// (okf_fmt_q2_0.hip): false, with nothing launched, where its shape or the
// device does not fit it.
bool launch_ffn_fused(okf_ctx *c, const FfnArgs &a);

// Whether the context's scratch may grow now: not after okf_ctx_reserve, and
// not while the stream is being captured into a graph (a synchronisation or
// hipMalloc would invalidate the capture).
inline bool can_grow(okf_ctx *c) {
    if (c->reserved) return false;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(c->stream, &cs) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return cs == hipStreamCaptureStatusNone;
}

// Grows one scratch buffer to at least `need` bytes (the stream is drained
// before an old buffer is freed).  Where it may not grow (can_grow) a call
// that needs more is an OKF_E_SHAPE, so nothing on a reserved or captured
// hot path allocates or synchronises.  A buffer that a captured graph holds
// (held) is not freed but kept until the context is destroyed, and its
// successor takes at least twice its bytes, so that the kept ones together
// are never more than the one in use.  `optional`: a failure records no HIP
// error (the caller runs without the buffer).
inline int grow_buf(okf_ctx *c, void **buf, size_t &bytes, bool &held, size_t need, bool zero, bool optional) {
    if (need <= bytes) return OKF_OK;
    if (!can_grow(c)) return OKF_E_SHAPE;
    hipError_t e = hipSuccess;
    size_t take = need;
    if (*buf) {
        e = hipStreamSynchronize(c->stream);
        if (e != hipSuccess) return optional ? ((void)hipGetLastError(), OKF_E_HIP) : hip_fail(c, e);
        if (held) {
            try {
                c->retired.push_back(*buf);
            } catch (const std::bad_alloc &) {
                return OKF_E_ARG;  // (the buffer stays as it is)
            }
            take = std::max(need, 2 * bytes);
        } else {
            (void)hipFree(*buf);
        }
        *buf = nullptr;
        bytes = 0;
        held = false;
    }
    e = hipMalloc(buf, take);
    if (e != hipSuccess && take > need) {
        (void)hipGetLastError();
        take = need;
        e = hipMalloc(buf, take);
    }
    if (e == hipSuccess && zero) e = hipMemset(*buf, 0, take);
    if (e != hipSuccess) {
        if (*buf) (void)hipFree(*buf);
        *buf = nullptr;
        return optional ? ((void)hipGetLastError(), OKF_E_HIP) : hip_fail(c, e);
    }
    bytes = take;
    return OKF_OK;
}

// split-tile partial sums and argmax pairs
inline int grow_part(okf_ctx *c, size_t need, bool optional = false) {
    return grow_buf(c, (void **)&c->part, c->part_bytes, c->part_held, need, false, optional);
}

// argmax row counters, zeroed when allocated (the kernel leaves them zero)
inline int grow_cnt(okf_ctx *c, size_t rows) {
    size_t bytes = c->cnt_n * sizeof(uint32_t);
    const int st = grow_buf(c, (void **)&c->cnt, bytes, c->cnt_held, rows * sizeof(uint32_t), true, false);
    c->cnt_n = bytes / sizeof(uint32_t);
    return st;
}

// the fp16 copy of a GEMM's activations: N K values
inline int grow_xh(okf_ctx *c, size_t need, bool optional = false) {
    return grow_buf(c, (void **)&c->xh, c->xh_bytes, c->xh_held, need, false, optional);
}

// ---------------------------------------------------------- tile GEMM plan
// How a tile GEMM runs: the few-token kernel (gemm_few_kernel, kind 0: fm
// row tiles and fn token tiles of 16 a workgroup) or the many-token one
// (gemm_many_kernel, kind 1: 16 fm rows x 128 fn tokens), and the K ranges
// (kper k each).
struct MmPlan {
    int kind, fm, fn;
    uint32_t ks, kper;
};

// The many-token instances: fm x fn accumulators of 4 registers a lane.
#define OKF_MANY(X) X(4, 1) X(5, 1) X(6, 1) X(8, 1) X(9, 1) X(4, 2) X(5, 2) X(6, 2) X(8, 2) X(9, 2) X(4, 3) X(5, 3) X(6, 3)
#define OKF_FEW(X) X(1, 1) X(2, 1) X(1, 2) X(2, 2) X(1, 4) X(2, 4)

inline bool mm_instance(int kind, int fm, int fn) {
#define OKF_IS(a, b) (fm == a && fn == b) ||
    return kind == 1 ? OKF_MANY(OKF_IS) false : kind == 0 ? OKF_FEW(OKF_IS) false : false;
#undef OKF_IS
}

// The plan with the least estimated time (us), from figures measured on
// MI355X over 300 x 768 .. 17408 x 5120 and 6 .. 1024 tokens (Q4_K, IQ4_NL):
//  many: a chunk takes fm (0.15 + 0.17 fn), a workgroup 5 besides, one
//    workgroup a CU at a time (so the tile height that just fills the CUs
//    wins: 17408 x 5120, N = 101: fm 5 38 us, 4 58, 8 58; N = 512: fm 9, fn 2
//    88 us, 8, 2 142), and its outputs, stored by all at once, 5 TB/s;
//  few: a wavefront's step takes 0.1 + w fm + 0.2 fn + 0.06 fm fn, times the
//    workgroups that share a CU, and 2.5 besides (6144 x 2048, N = 19: 7.7 us
//    against 11.1 for many; N = 48: 10.3 against 13.4); w: 0.25, more for the
//    formats whose pieces take many loads; past one workgroup a CU no less than
//    0.55 fm fn each, the sum of its wavefronts' tiles (IQ4_NL 151936 x 1024, N = 33:
//    fm 2, fn 4 108 us, many with fm 8 72; Q4_K 65536 x 512 36 and 21);
//  K ranges: the partial tiles written and read at 5 TB/s, and a launch.
// From 256 tokens on the formats but Q4_K take only many, whose sums are in
// gemm_mfma_kernel's order (few takes K in another order within 128).
// room: bytes there are for partial tiles; a plan takes as many K ranges as fit
// (without room for two, one range, whose best tile is another: Q4_K 5120 x
// 17408, N = 64, 64 workgroups of the K-split plan's tile 113 us, the one-range plan 56).
inline MmPlan plan_mm(const okf_ctx *c, int type, uint32_t K, uint32_t M, uint32_t N, size_t room = SIZE_MAX) {
    const uint32_t cus = c->cus ? c->cus : 256;
    auto up = [](uint64_t a, uint64_t b) { return (a + b - 1) / b; };
    MmPlan p{};
    double best = 0;
    const double w = type == Q6_K ? 0.75 : type == Q8_0 ? 0.6 : dq_fast(type) ? 0.25 : 0.9;
    const int *force = c->gemm_plan;  // (measurements and tests)
    auto consider = [&](int kind, int fm, int fn, uint32_t ks) {
        if (force[1] && (kind != force[0] || fm != force[1] || fn != force[2])) return;
        if (force[1]) ks = (uint32_t)force[3];
        if (!kind && up(N, 16 * fn) > 65535) return;  // (the grid's second dimension; many has all tiles in the first)
        ks = (uint32_t)std::min<uint64_t>(ks, std::max<uint64_t>(1, room / ((uint64_t)N * M * sizeof(float))));
        const uint32_t unit = kind ? MC_BK : 128, steps = (uint32_t)up(K, unit);
        const uint32_t per = (uint32_t)up(steps, std::max(1u, std::min(ks, steps)));
        ks = (uint32_t)up(steps, per);
        const uint64_t wgs = up(M, 16 * fm) * up(N, (kind ? 128 : 16) * fn) * ks;
        double t = (double)N * M * 4 / 5e6 + (ks > 1 ? 2.5 + (double)ks * N * M * 8 / 5e6 : 0);
        if (kind) t += (double)up(wgs, cus) * (per * fm * (0.15 + 0.17 * fn) + 5);
        else {
            const double wg = (double)up(per, 4) * (0.1 + w * fm + 0.2 * fn + 0.06 * fm * fn), more = (double)wgs / cus - 1;
            t += 2.5 + wg + std::max(0.0, more) * std::max(wg, 0.55 * fm * fn);
        }
        if (best == 0 || t < best) {
            best = t;
            p = MmPlan{kind, fm, fn, ks, per * unit};
        }
    };
    if (force[1] || (c->gemm_ks == 0 && (N < 256 || type == Q4_K))) {
#define OKF_CONSIDER(a, b)                      \
    for (uint32_t ks = 1; ks <= (c->gemm_split ? 4u : 1u); ks *= 2) consider(0, a, b, ks);
        OKF_FEW(OKF_CONSIDER)
#undef OKF_CONSIDER
    }
    auto many = [&](int fm, int fn) {
        const uint64_t tiles = up(M, 16 * fm) * up(N, 128 * fn);
        if (c->gemm_ks > 0) return consider(1, fm, fn, (uint32_t)c->gemm_ks);
        consider(1, fm, fn, 1);
        if (!c->gemm_split) return;
        // as many K ranges as fill one or two rounds of the CUs
        for (uint32_t r = 1; r <= 2; r++)
            if (r * cus / tiles > 1) consider(1, fm, fn, (uint32_t)(r * cus / tiles));
    };
#define OKF_CONSIDER(a, b) many(a, b);
    OKF_MANY(OKF_CONSIDER)
#undef OKF_CONSIDER
    return p;  // (OKF_GEMM_PLAN is checked against the instances when it is read)
}

// Marks the scratch buffers that a call hands to its launches, where they are
// being captured into a graph: the graph holds their addresses (grow_buf).
inline void note_capture(okf_ctx *c, bool xh, bool part, bool cnt) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(c->stream, &cs) != hipSuccess) {
        (void)hipGetLastError();
    } else if (cs != hipStreamCaptureStatusNone) {
        c->xh_held |= xh;
        c->part_held |= part;
        c->cnt_held |= cnt;
    }
}

template <int F>
int launch_gemm(okf_ctx *c, const uint8_t *W, uint64_t rb, uint32_t K, uint32_t M, const float *X,
                uint32_t N, float *Y) {
    // fp16 activations, converted once per call into the context's buffer
    // (as octets: x_to_octets_kernel)
    const int st = c->gemm_xh || F == Q4_K ? grow_xh(c, (size_t)N * K * sizeof(_Float16), F != Q4_K) : OKF_E_SHAPE;
    if (st && F == Q4_K) return st;
    // the K ranges' partial tiles, added in K order by gemm_ksum_kernel
    auto partials = [&](uint32_t ks) { return grow_part(c, (size_t)ks * N * M * sizeof(float), true) == OKF_OK; };
    MmPlan p = plan_mm(c, F, K, M, N);
    if (st && c->gemm_xh) {
        // no room for X: gemm_mfma_kernel, which rounds X per tile.  A grid
        // of fewer than two tiles a CU (small M or N) takes K in ks ranges of
        // whole 64-steps; without room for their partial tiles, one range.
        const uint32_t tiles = ((N + GB_N - 1) / GB_N) * ((M + GB_M - 1) / GB_M), steps = (K + GB_K - 1) / GB_K;
        p.ks = 1;
        if (c->gemm_split != 0 && tiles < 2 * c->cus) {
            p.ks = c->gemm_split > 1 ? (uint32_t)c->gemm_split : (2 * c->cus + tiles - 1) / tiles;
            p.ks = std::max(1u, std::min(p.ks, steps / 4));
        }
        p.kper = (steps + p.ks - 1) / p.ks * GB_K;
        p.ks = (K + p.kper - 1) / p.kper;
        if (p.ks > 1 && !partials(p.ks)) p.ks = 1, p.kper = steps * GB_K;
    } else if (p.ks > 1 && !partials(p.ks)) {
        // (a reserved context, a stream being captured, or no memory: planned
        // again for the room that there is)
        p = plan_mm(c, F, K, M, N, c->part_bytes);
    }
    const uint32_t ks = p.ks, kper = p.kper;
    float *part = ks > 1 ? c->part : nullptr;
    note_capture(c, !st, part != nullptr, false);
    const u32x4 *tab = dq_tab_rows<F>() ? c->tab8 : nullptr;
    if (st) {
        if constexpr (F != Q4_K) {
            dim3 grid((N + GB_N - 1) / GB_N, (M + GB_M - 1) / GB_M, ks);
            hipLaunchKernelGGL((gemm_mfma_kernel<F>), grid, dim3(256), 0, c->stream, W, rb, K, M, X, N, Y, c->grid,
                               c->grids, kper, part);
        }
    } else {
        half8 *xt = (half8 *)c->xh;
        hipLaunchKernelGGL(x_to_octets_kernel, dim3((N + 15) / 16, (K / 8 + 63) / 64), dim3(256), 0, c->stream, X, N, K / 8,
                           xt);
        if (p.kind == 0) {
            auto go = [&](auto fmc, auto fnc) {
                constexpr int FM = decltype(fmc)::value, FN = decltype(fnc)::value;
                dim3 grid((M + 16 * FM - 1) / (16 * FM), (N + 16 * FN - 1) / (16 * FN), ks);
                hipLaunchKernelGGL((gemm_few_kernel<F, FM, FN, 4>), grid, dim3(256), 0, c->stream, W, rb, K, M, xt, N, Y,
                                   kper / 128, part, tab, c->grid, c->grids);
            };
#define OKF_GO(a, b) \
    if (p.fm == a && p.fn == b) go(std::integral_constant<int, a>{}, std::integral_constant<int, b>{});
            OKF_FEW(OKF_GO)
        } else {
            auto go = [&](auto fmc, auto fnc) {
                constexpr int FM = decltype(fmc)::value, FN = decltype(fnc)::value;
                const MmTiles mt{(M + 16 * FM - 1) / (16 * FM), (N + 128 * FN - 1) / (128 * FN), kper / MC_BK};
                hipLaunchKernelGGL((gemm_many_kernel<F, FM, FN>), dim3(mt.tiles_m * mt.tiles_n, 1, ks), dim3(512), 0,
                                   c->stream, W, rb, K, M, xt, N, Y, mt, part, tab, c->grid, c->grids);
            };
            OKF_MANY(OKF_GO)
#undef OKF_GO
        }
    }
    if (part) {
        const uint64_t nm = (uint64_t)N * M;
        hipLaunchKernelGGL(gemm_ksum_kernel, dim3((uint32_t)((nm + 1023) / 1024)), dim3(256), 0, c->stream,
                           (const float *)part, Y, nm, ks, (uint32_t)(nm % 4 == 0 && aligned16(Y)));
    }
    return OKF_OK;
}

template <int F>
void launch_dequant(okf_ctx *c, const uint8_t *row, uint32_t n, float *out) {
    const uint32_t units = n / 32;
    hipLaunchKernelGGL((dequant_row_kernel<F>), dim3((units + 255) / 256), dim3(256), 0, c->stream,
                       row, units, out, c->grid, c->grids);
}

template <int F>
void launch_embed(okf_ctx *c, const uint8_t *W, uint64_t rb, uint32_t K, uint32_t M,
                  const int32_t *ids, uint32_t N, float *out) {
    const uint32_t upr = K / 32, units = N * upr;
    hipLaunchKernelGGL((embed_batch_kernel<F>), dim3((units + 255) / 256), dim3(256), 0, c->stream, W,
                       rb, M, ids, upr, units, out, c->grid, c->grids);
}

// Every format with kernels here, for the per-format instantiations.
#define OKF_FOR_EACH_FORMAT(X)                                                                           \
    X(Q8_0) X(Q2_0) X(Q4_K) X(Q4_0) X(IQ4_NL) X(Q5_K) X(Q6_K) X(IQ4_XS) X(IQ2_XS) X(IQ2_S) X(IQ3_XXS)     \
    X(IQ3_S) X(IQ1_S) X(IQ1_M) X(Q2_K) X(Q3_K) X(F32) X(F16) X(BF16) X(IQ2_XXS)

#define OKF_LAUNCHERS(EXT, F)                                                                            \
    EXT template void launch_gemv<F>(okf_ctx *, const GemvCall *, int, uint64_t, uint32_t, uint32_t);    \
    EXT template void launch_gemv_pair<F>(okf_ctx *, const GemvCall *, uint64_t, uint32_t);               \
    EXT template int launch_gemm<F>(okf_ctx *, const uint8_t *, uint64_t, uint32_t, uint32_t, const float *, \
                                    uint32_t, float *);                                                  \
    EXT template void launch_dequant<F>(okf_ctx *, const uint8_t *, uint32_t, float *);                  \
    EXT template void launch_embed<F>(okf_ctx *, const uint8_t *, uint64_t, uint32_t, uint32_t,          \
                                      const int32_t *, uint32_t, float *);
#define OKF_EXTERN(F) OKF_LAUNCHERS(extern, F)
#define OKF_INSTANTIATE(F) OKF_LAUNCHERS(, F)

}  // namespace okf_impl
