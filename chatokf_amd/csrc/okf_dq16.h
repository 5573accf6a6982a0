// okf_dq16.h -- one lane's 32 weights as fp16, for the matrix-core GEMMs.
//
// A lane takes a "piece" of a row: 32 weights whose packed bytes it can load
// with one or two wide loads.  Piece u of a row gives four octets (8
// consecutive weights each, the k of one lane of an MFMA operand); octet i of
// piece u is weights 8 dq_octet<F>(u, i) .. + 7 of the row.  The loads
// (DqRaw) are apart from the conversion (dq_piece), so that the bytes of a
// later step are in flight while a step computes.
//
// Every weight is rounded to fp16 once, from a product that is exact before
// that, so it is the fp16 rounding of the weight that decode_unit gives: an exact
// small integer in fp16 times an fp16 scale (dq_mul: Q8_0, Q2_0, Q4_0, IQ4_NL), or
// fma(q, a, o) with a, o in fp32 (dq_pair, v_fma_mixlo_f16 / v_fma_mixhi_f16; Q4_K
// and Q5_K: the fp32 sum has one more rounding of 2^-24).  Infinite scales: dq_inf.
#pragma once
#include <type_traits>

#include "okf_common.h"
#include "okf_decode.h"
#include "okf_gemv.h"

namespace okf {

// the formats with loads and conversions of their own; the others decode
// from memory at conversion time (DqRaw keeps the row)
__host__ __device__ constexpr bool dq_fast(int f) {
    return f == Q8_0 || f == Q2_0 || f == Q4_0 || f == IQ4_NL || f == Q4_K || f == Q5_K || f == Q6_K ||
           f == IQ4_XS || f == IQ2_XXS;
}
// 8-byte table entries a conversion reads from LDS (IQ2_XXS: the grid and
// sign entries of Compute<IQ2_XXS>)
template <int F>
__host__ __device__ constexpr uint32_t dq_tab_rows() {
    return F == IQ2_XXS ? 384 : 0;
}

// Octet (8 weights) index in the row of output i of piece u.
//  Q4_K, Q5_K: piece j of a superblock is 16 code bytes, half h = j % 2 of
//    code group g = j / 2: low nibbles are weights 64 g + 16 h .., high ones
//    32 further.
//  Q6_K: piece j is code bytes 8 (j % 4) .. + 7 of half n = j / 4: octet i is
//    weights 128 n + 32 i + 8 (j % 4) ..
template <int F>
__device__ __forceinline__ uint32_t dq_octet(uint32_t u, int i) {
    if constexpr (F == Q4_K || F == Q5_K) return (u & ~7u) * 4 + 8 * ((u & 7) >> 1) + 2 * (u & 1) + (i & 1) + 4 * (i >> 1);
    else if constexpr (F == Q6_K) return (u & ~7u) * 4 + 16 * ((u >> 2) & 1) + 4 * i + (u & 3);
    else return 4 * u + i;
}

template <int F>
struct DqRaw {
    const uint8_t *row;
    uint32_t u;
};
template <>
struct DqRaw<Q8_0> {
    uint32_t d;
    u32x4 q0, q1;
};
template <>
struct DqRaw<Q2_0> {
    uint32_t d;
    uint2 q;
};
template <>
struct DqRaw<Q4_0> {
    uint32_t d;
    u32x4 q;
};
template <>
struct DqRaw<IQ4_NL> {
    uint32_t d;
    u32x4 q;
};
template <>
struct DqRaw<Q4_K> {
    u32x4 hdr, q;
};
template <>
struct DqRaw<Q5_K> {
    u32x4 hdr, q, qh;
};
template <>
struct DqRaw<Q6_K> {
    uint32_t d;
    uint2 lo, hi, qh, sc;
};
template <>
struct DqRaw<IQ4_XS> {
    uint2 hdr;
    u32x4 q;
};
template <>
struct DqRaw<IQ2_XXS> {
    uint32_t d;
    uint2 a;
};

template <int F>
__device__ __forceinline__ void dq_load(const uint8_t *row, uint32_t u, DqRaw<F> &r) {
    if constexpr (F == Q8_0) {
        const uint8_t *b = row + (uint64_t)u * 34;
        r.d = ldu<uint16_t>(b);
        r.q0 = ldu<u32x4>(b + 2);
        r.q1 = ldu<u32x4>(b + 18);
    } else if constexpr (F == Q2_0) {
        const uint8_t *b = row + (uint64_t)(u >> 2) * 34;
        r.d = ldu<uint16_t>(b);
        r.q = ldu<uint2>(b + 2 + (u & 3) * 8);
    } else if constexpr (F == Q4_0 || F == IQ4_NL) {
        const uint8_t *b = row + (uint64_t)u * 18;
        r.d = ldu<uint16_t>(b);
        r.q = ldu<u32x4>(b + 2);
    } else if constexpr (F == Q4_K) {
        const uint8_t *b = row + (uint64_t)(u >> 3) * 144;
        r.hdr = *(const u32x4 *)b;
        r.q = *(const u32x4 *)(b + 16 + 16 * (u & 7));
    } else if constexpr (F == Q5_K) {
        const uint8_t *b = row + (uint64_t)(u >> 3) * 176;
        r.hdr = ldu<u32x4>(b);
        r.qh = ldu<u32x4>(b + 16 + 16 * (u & 1));
        r.q = ldu<u32x4>(b + 48 + 16 * (u & 7));
    } else if constexpr (F == Q6_K) {
        const uint8_t *b = row + (uint64_t)(u >> 3) * 210;
        const uint32_t n = (u >> 2) & 1, l = 8 * (u & 3);
        r.d = ldu<uint16_t>(b + 208);
        r.sc = ldu<uint2>(b + 192 + 8 * n);
        r.lo = ldu<uint2>(b + 64 * n + l);
        r.hi = ldu<uint2>(b + 64 * n + 32 + l);
        r.qh = ldu<uint2>(b + 128 + 32 * n + l);
    } else if constexpr (F == IQ4_XS) {
        const uint8_t *b = row + (uint64_t)(u >> 3) * 136;
        r.hdr = ldu<uint2>(b);
        r.q = ldu<u32x4>(b + 8 + 16 * (u & 7));
    } else if constexpr (F == IQ2_XXS) {
        const uint8_t *b = row + (uint64_t)(u >> 3) * 66;
        r.d = ldu<uint16_t>(b);
        r.a = ldu<uint2>(b + 2 + 8 * (u & 7));
    } else {
        r.row = row;
        r.u = u;
    }
}

// two fp16 in a dword, each fma(q, a, o) rounded once
__device__ __forceinline__ uint32_t dq_pair(half2v q, float a, float o) {
    const half2v r = {(_Float16)fmaf((float)q[0], a, o), (_Float16)fmaf((float)q[1], a, o)};
    return __builtin_bit_cast(uint32_t, r);
}
// Two exact codes by a scale that is itself an fp16 value: one packed
// multiplication rounds the exact product once (the bits of dq_pair).
__device__ __forceinline__ uint32_t dq_mul(half2v q, _Float16 d) {
    return __builtin_bit_cast(uint32_t, q * half2v{d, d});
}
__device__ __forceinline__ half2v dq_h2(uint32_t v) { return __builtin_bit_cast(half2v, v); }
// 8 unsigned bytes (dwords b0, b1) less C, exactly in fp16 through 1024 + byte,
// each pair through f; C < 0: as 1024 + byte
template <int C, class Fn>
__device__ __forceinline__ half8 dq_bytes(uint32_t b0, uint32_t b1, Fn f) {
    auto q = [&](uint32_t b, uint32_t sel) {
        const half2v p = dq_h2(perm(0x64646464u, b, sel));
        if constexpr (C < 0) return f(p);
        else return f(p + half2v{(_Float16)(-1024.0f - C), (_Float16)(-1024.0f - C)});
    };
    return __builtin_bit_cast(half8, uint4{q(b0, 0x04010400u), q(b0, 0x04030402u), q(b1, 0x04010400u),
                                           q(b1, 0x04030402u)});
}
// 8 nibbles (one per byte of b0, b1) exactly in fp16 through
// v_cvt_scalef32_pk_f16_fp8 (a nibble in an e4m3 byte is q 2^-9), each pair through f
template <class Fn>
__device__ __forceinline__ half8 dq_nibbles(uint32_t b0, uint32_t b1, Fn f) {
    return __builtin_bit_cast(half8, uint4{f(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(b0, 512.0f, false)),
                                           f(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(b0, 512.0f, true)),
                                           f(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(b1, 512.0f, false)),
                                           f(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(b1, 512.0f, true))});
}

// An infinite block scale gives +-inf, and NaN for a zero code, as in the decoders,
// where the codes meet it without an offset.  IQ4_XS and IQ2_XXS, whose sub-block
// scales are no fp16 values, keep the offset in the fma (a q + o with o = -C a, exact:
// a has at most 18 significant bits), which would give NaN for all: their scale is
// then 1 (dq_d1) and the codes are multiplied by it after, behind a branch that a
// wavefront of finite scales passes by.  Measured against the offset in every
// fma and no guard, the mean over 1000 x 1024 to 5120 x 17408 and 13 to 512
// tokens: the packed multiplication Q8_0 0.981, Q2_0 0.957, Q4_0 0.975, IQ4_NL 0.968;
// the branch IQ4_XS and IQ2_XXS 1.000 (offset taken off the codes: 1.020, 1.027); Q6_K
// with the branch 1.033, with the offset taken off 1.006.
__device__ __forceinline__ float dq_d1(float d) { return __builtin_isinf(d) ? 1.0f : d; }
__device__ __forceinline__ void dq_inf(float d, half8 (&h)[4]) {
    if (__any(__builtin_isinf(d))) {
        const float s = __builtin_isinf(d) ? d : 1.0f;
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int e = 0; e < 8; e++) h[i][e] = (_Float16)((float)h[i][e] * s);
    }
}

// the IQ4 levels + 128 as unsigned bytes (IQ4Levels' lookup)
__host__ __device__ constexpr uint32_t iq4_lvu4(int i) { return iq4_lv4(i) ^ 0x80808080u; }
__device__ __forceinline__ uint32_t iq4_levels_u(uint32_t nib) {
    constexpr uint32_t T0 = iq4_lvu4(0), T1 = iq4_lvu4(4), T2 = iq4_lvu4(8), T3 = iq4_lvu4(12);
    const uint32_t sel = nib & 0x07070707u;
    const uint32_t lo = perm(T1, T0, sel), hi = perm(T3, T2, sel);
    return perm(hi, lo, ((nib >> 1) & 0x04040404u) | 0x03020100u);
}

// Piece r as fp16: h[i] = octet dq_octet(u, i).  tab: the LDS tables
// (dq_tab_rows), grid / gt: the device-memory grids of the formats that
// decode from memory.
template <int F>
__device__ __forceinline__ void dq_piece(const DqRaw<F> &r, uint32_t u, half8 (&h)[4], const uint2 *tab,
                                         const uint2 *grid, const uint8_t *gt) {
    if constexpr (F == Q8_0) {
        const _Float16 d = __builtin_bit_cast(_Float16, (uint16_t)r.d);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const u32x4 &q = i < 2 ? r.q0 : r.q1;
            h[i] = dq_bytes<128>(q[2 * (i & 1)] ^ 0x80808080u, q[2 * (i & 1) + 1] ^ 0x80808080u,
                                 [&](half2v v) { return dq_mul(v, d); });
        }
    } else if constexpr (F == Q2_0) {  // code j at bits 2 (j % 16) of dword j / 16
        const _Float16 d = __builtin_bit_cast(_Float16, (uint16_t)r.d);
        const half2v m = {(_Float16)-1025.0f, (_Float16)-1025.0f};
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const uint32_t dw = s ? r.q.y : r.q.x;
            const uint32_t f0 = dw & 0x03030303u, f1 = (dw >> 2) & 0x03030303u;
            const uint32_t f2 = (dw >> 4) & 0x03030303u, f3 = (dw >> 6) & 0x03030303u;
            uint32_t p[8];
#pragma unroll
            for (int k = 0; k < 4; k++) {  // weights 4 k + {0, 1 | 2, 3}: byte k of f0 f1 | f2 f3
                const uint32_t sel = (uint32_t)k | 0x0C00u | (uint32_t)(4 + k) << 16 | 0x0C000000u;
                p[2 * k] = perm(f1, f0, sel) | 0x64006400u;
                p[2 * k + 1] = perm(f3, f2, sel) | 0x64006400u;
            }
#pragma unroll
            for (int k = 0; k < 2; k++)
                h[2 * s + k] = __builtin_bit_cast(
                    half8, uint4{dq_mul(dq_h2(p[4 * k]) + m, d), dq_mul(dq_h2(p[4 * k + 1]) + m, d),
                                 dq_mul(dq_h2(p[4 * k + 2]) + m, d), dq_mul(dq_h2(p[4 * k + 3]) + m, d)});
        }
    } else if constexpr (F == Q4_0) {  // byte j: weight j (low nibble), j + 16 (high)
        const _Float16 d = __builtin_bit_cast(_Float16, (uint16_t)r.d);
        const half2v m = {(_Float16)-8.0f, (_Float16)-8.0f};
        auto f = [&](half2v v) { return dq_mul(v + m, d); };
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t v0 = r.q[2 * (i & 1)], v1 = r.q[2 * (i & 1) + 1];
            h[i] = i < 2 ? dq_nibbles(v0 & 0x0F0F0F0Fu, v1 & 0x0F0F0F0Fu, f)
                         : dq_nibbles((v0 >> 4) & 0x0F0F0F0Fu, (v1 >> 4) & 0x0F0F0F0Fu, f);
        }
    } else if constexpr (F == IQ4_NL || F == IQ4_XS) {
        auto put = [&](auto cc, auto f) {
            constexpr int C = decltype(cc)::value;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t v0 = r.q[2 * (i & 1)], v1 = r.q[2 * (i & 1) + 1];
                h[i] = i < 2 ? dq_bytes<C>(iq4_levels_u(v0 & 0x0F0F0F0Fu), iq4_levels_u(v1 & 0x0F0F0F0Fu), f)
                             : dq_bytes<C>(iq4_levels_u((v0 >> 4) & 0x0F0F0F0Fu), iq4_levels_u((v1 >> 4) & 0x0F0F0F0Fu), f);
            }
        };
        if constexpr (F == IQ4_NL) {
            const _Float16 d = __builtin_bit_cast(_Float16, (uint16_t)r.d);
            put(std::integral_constant<int, 128>{}, [&](half2v v) { return dq_mul(v, d); });
        } else {
            const uint32_t ib = u & 7, sh = r.hdr.x >> 16, sl = r.hdr.y >> (4 * ib);
            const float d = h2f(r.hdr.x & 0xFFFF);
            const float a = dq_d1(d) * (float)((int)((sl & 0xF) | (((sh >> (2 * ib)) & 3) << 4)) - 32), o = -1152.0f * a;
            put(std::integral_constant<int, -1>{}, [&](half2v v) { return dq_pair(v, a, o); });
            dq_inf(d, h);
        }
    } else if constexpr (F == Q4_K || F == Q5_K) {
        const uint32_t j = u & 7, g = j >> 1;
        // the 6-bit scales and mins of sub-blocks 2 g, 2 g + 1
        const uint32_t s1 = r.hdr[1], s2 = r.hdr[2], s3 = r.hdr[3], sh = 16 * (g & 1);
        uint32_t sc, mn;
        if (g < 2) {
            sc = (s1 >> sh) & 0x3F3Fu;
            mn = (s2 >> sh) & 0x3F3Fu;
        } else {
            sc = ((s3 >> sh) & 0x0F0Fu) | ((s1 >> (sh + 2)) & 0x3030u);
            mn = ((s3 >> (sh + 4)) & 0x0F0Fu) | ((s2 >> (sh + 2)) & 0x3030u);
        }
        const float d = h2f(r.hdr[0] & 0xFFFF), dmin = -h2f(r.hdr[0] >> 16);
        const float a0 = d * (float)(sc & 0xFF), a1 = d * (float)(sc >> 8);
        const float o0 = dmin * (float)(mn & 0xFF), o1 = dmin * (float)(mn >> 8);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t v0 = i < 2 ? r.q[2 * (i & 1)] : r.q[2 * (i & 1)] >> 4;
            const uint32_t v1 = i < 2 ? r.q[2 * (i & 1) + 1] : r.q[2 * (i & 1) + 1] >> 4;
            const float a = i < 2 ? a0 : a1, o = i < 2 ? o0 : o1;
            if constexpr (F == Q4_K) {
                h[i] = dq_nibbles(v0 & 0x0F0F0F0Fu, v1 & 0x0F0F0F0Fu, [&](half2v v) { return dq_pair(v, a, o); });
            } else {
                // the fifth bit: bit 2 g (+ 1) of the qh byte
                const uint32_t t = 2 * g + (i >> 1);
                const uint32_t b0 = (v0 & 0x0F0F0F0Fu) | (((r.qh[2 * (i & 1)] >> t) & 0x01010101u) << 4);
                const uint32_t b1 = (v1 & 0x0F0F0F0Fu) | (((r.qh[2 * (i & 1) + 1] >> t) & 0x01010101u) << 4);
                const half2v m = {(_Float16)-1024.0f, (_Float16)-1024.0f};
                auto pr = [&](uint32_t b, uint32_t sel) {
                    return dq_pair(__builtin_bit_cast(half2v, perm(0x64646464u, b, sel)) + m, a, o);
                };
                h[i] = __builtin_bit_cast(half8, uint4{pr(b0, 0x04010400u), pr(b0, 0x04030402u), pr(b1, 0x04010400u),
                                                       pr(b1, 0x04030402u)});
            }
        }
    } else if constexpr (F == Q6_K) {
        const float d = h2f(r.d);
        const uint32_t is = (u >> 1) & 1;  // scale 2 i + is of the half's 8
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint2 l = (i & 1) ? r.hi : r.lo;
            const int s = (int8_t)((i < 2 ? r.sc.x : r.sc.y) >> (16 * (i & 1) + 8 * is));
            const float a = d * (float)s;
            const uint32_t b0 = ((l.x >> (4 * (i >> 1))) & 0x0F0F0F0Fu) | (((r.qh.x >> (2 * i)) & 0x03030303u) << 4);
            const uint32_t b1 = ((l.y >> (4 * (i >> 1))) & 0x0F0F0F0Fu) | (((r.qh.y >> (2 * i)) & 0x03030303u) << 4);
            h[i] = dq_bytes<32>(b0, b1, [&](half2v v) { return dq_pair(v, a, 0.0f); });
        }
    } else if constexpr (F == IQ2_XXS) {
        const float a = dq_d1(h2f(r.d)) * (0.5f + (float)(r.a.y >> 28)) * 0.25f, o = -1152.0f * a;
        // {8, 25, 43 | -8, -25, -43} + 128 (Compute<IQ2_XXS>'s selection)
        constexpr uint32_t POS = IQ2_POS ^ 0x80808080u, NEG = IQ2_NEG ^ 0x80808080u;
#pragma unroll
        for (int l = 0; l < 4; l++) {
            const uint2 gv = tab[(r.a.x >> (8 * l)) & 0xFF];
            const uint2 sg = tab[256 + ((r.a.y >> (7 * l)) & 127)];
            h[l] = dq_bytes<-1>(perm(NEG, POS, gv.x + sg.x - 0x03020100u), perm(NEG, POS, gv.y + sg.y - 0x03020100u),
                                [&](half2v v) { return dq_pair(v, a, o); });
        }
        dq_inf(h2f(r.d), h);
    } else {
        float w[32];
        decode_unit<F>(r.row, r.u, w, grid, gt);
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int e = 0; e < 8; e++) h[i][e] = (_Float16)w[8 * i + e];
    }
}

}  // namespace okf
