// The file's blocks of the ggml types without kernel planes, read value by value or a 32-value unit at a time: shared by
// the exact path's rebuild (mbq_kernels.hip) and its fused products (mbq_raw.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mbq_device.h"
#include "mbq_layout.h"

namespace mbq {

// ---------------------------------------------------------------------------- raw dequant, the other ggml types
// The exact path's rebuild for the ggml types that have no kernel planes here (reference src/mashbox/ops/reference.py,
// the line ranges at each type below). Every value is exact or rounded once, as in the reference: a product of an fp16
// scale and a small integer is exact in float32, so d * q + m (Q4_1, Q5_1) and dl * q - ml (Q2_K) round once whether
// or not the compiler fuses them; IQ4_XS's (d * s) * k rounds once in the second product, in that order.
__device__ __forceinline__ uint32_t le16(const uint8_t* p) { return (uint32_t)p[0] | ((uint32_t)p[1] << 8); }
__device__ __forceinline__ uint32_t le32(const uint8_t* p) { return le16(p) | (le16(p + 2) << 16); }
// value i (0..31) of a 32-value block's 16 nibble bytes: low nibbles first, then the high ones
__device__ __forceinline__ uint32_t nib32(const uint8_t* qs, int i) { return (qs[i & 15] >> (4 * (i >> 4))) & 15u; }
// ggml's kvalues_iq4nl (reference :348) and the FP4 (E2M1) values doubled, kvalues_mxfp4 (reference :195)
static __constant__ float kIQ4[16] = {-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113};
static __constant__ float kFP4[16] = {0, 1, 2, 3, 4, 6, 8, 12, 0, -1, -2, -3, -4, -6, -8, -12};

// MXFP4 (reference :198-219): k * 2^(e - 128) with the float32 bits built from integers, so results below the normal
// range are exact subnormals, results past it inf, and zero codes +0
__device__ __forceinline__ float mxfp4_value(uint32_t e, uint32_t q) {
    const uint32_t c = q & 7u;
    const int odd = (int)((0x31313110u >> (4 * c)) & 15u);     // |k| = odd * 2^p for c = 0..7: odd 0 1 1 3 1 3 1 3,
    const int p = (int)((0x23120100u >> (4 * c)) & 15u);       //                                 p   0 0 1 0 2 1 3 2
    if (odd == 0) return 0.f;
    const int x = p + (int)e - 128, E = odd == 3 ? x + 1 : x;
    uint32_t bits;
    if (E > 127) bits = 0x7F800000u;
    else if (E < -126) bits = (uint32_t)odd << (x + 149);                                // x >= -128: a shift of 21-22
    else bits = ((uint32_t)(E + 127) << 23) | (odd == 3 ? 1u << 22 : 0u);
    return __uint_as_float(bits | (q >= 8 ? 0x80000000u : 0u));
}

// NVFP4's block scale (reference :222-227): unsigned E4M3 of bits 0-6 (bias 7), halved; the bytes 0x00 and 0x7F give 0
__device__ __forceinline__ float ue4m3_half(uint32_t x) {
    if (x == 0u || x == 0x7Fu) return 0.f;
    const uint32_t e = (x >> 3) & 15u;
    const float man = (float)(x & 7u);
    const float raw = e == 0 ? man * 0x1p-9f : (1.f + man * 0.125f) * __uint_as_float((e + 120u) << 23);
    return raw * 0.5f;
}

// TQ1_0's code of value v (reference :176-185): the base-3 digit k of a byte, ((byte * 3^k mod 256) * 3) >> 8, over
// bytes 0-31 (values 0-159, k = v / 32), 32-47 (values 160-239) and 48-51 (values 240-255)
__device__ __forceinline__ int tq1_code(const uint8_t* b, int v) {
    int k, byte;
    if (v < 160) k = v >> 5, byte = b[v & 31];
    else if (v < 240) k = (v - 160) >> 4, byte = b[32 + ((v - 160) & 15)];
    else k = (v - 240) >> 2, byte = b[48 + ((v - 240) & 3)];
    const int pw = k == 0 ? 1 : k == 1 ? 3 : k == 2 ? 9 : k == 3 ? 27 : 81;
    return ((((byte * pw) & 255) * 3) >> 8) - 1;
}

// the alignment every block start of type T has when the blocks start at an address of that alignment: the largest
// power of two (at most 4) dividing the block bytes (Q2_K 84, Q4_1 20, Q5_1 24, IQ4_XS 136, NVFP4 36, F32: 4; Q3_K
// 110, Q5_0 22, IQ4_NL 18, TQ1_0 54, TQ2_0 66, F16, BF16: 2; MXFP4 17: 1). Told to the compiler, it lets it merge the
// byte reads of a block into wider loads.
template <int T>
__host__ __device__ constexpr int raw_align() { return raw_block_align(T); }
static_assert(raw_block_align(T_Q2_K) == 4 && raw_block_align(T_Q3_K) == 2 && raw_block_align(T_MXFP4) == 1 &&
              raw_block_align(T_F32) == 4 && raw_block_align(T_BF16) == 2, "block alignments");
template <int T>
__device__ __forceinline__ const uint8_t* blk(const uint8_t* p) {
    return static_cast<const uint8_t*>(__builtin_assume_aligned(p, raw_align<T>()));
}

// Values 32u .. 32u + 31 of one weight row in the file's blocks of type T (row: the row's first byte, aligned to
// raw_align<T>()): a block of the 32-value types, half an NVFP4 block, a 32-value group of a 256-value super-block; for
// the float types (one value per block) 32 consecutive values
template <int T>
__device__ __forceinline__ void raw_unit(const uint8_t* __restrict__ row, int u, float v[32]) {
    if constexpr (T == T_F32 || T == T_F16 || T == T_BF16) {            // reference :372-381
        constexpr int ES = T == T_F32 ? 4 : 2;
        const uint8_t* p = blk<T>(row + (int64_t)ES * 32 * u);
        for (int i = 0; i < 32; ++i)
            v[i] = T == T_F32 ? __uint_as_float(le32(p + 4 * i)) : T == T_F16 ? f16f(le16(p + 2 * i))
                                                                       : __uint_as_float(le16(p + 2 * i) << 16);
    } else if constexpr (T == T_Q4_1) {                                  // reference :73-77
        const uint8_t* b = blk<T>(row + (int64_t)u * 20);
        const float d = f16f(le16(b)), m = f16f(le16(b + 2));
        for (int i = 0; i < 32; ++i) v[i] = d * (float)nib32(b + 4, i) + m;
    } else if constexpr (T == T_Q5_0 || T == T_Q5_1) {                   // reference :85-98
        constexpr bool ONE = T == T_Q5_1;
        const uint8_t* b = blk<T>(row + (int64_t)u * (ONE ? 24 : 22));
        const float d = f16f(le16(b)), m = ONE ? f16f(le16(b + 2)) : 0.f;
        const uint32_t qh = le32(b + (ONE ? 4 : 2));
        const uint8_t* qs = b + (ONE ? 8 : 6);
        for (int i = 0; i < 32; ++i) {
            const int q = (int)(nib32(qs, i) | (((qh >> i) & 1u) << 4));
            v[i] = ONE ? d * (float)q + m : d * (float)(q - 16);
        }
    } else if constexpr (T == T_IQ4_NL) {                                // reference :351-356
        const uint8_t* b = blk<T>(row + (int64_t)u * 18);
        const float d = f16f(le16(b));
        for (int i = 0; i < 32; ++i) v[i] = d * kIQ4[nib32(b + 2, i)];
    } else if constexpr (T == T_MXFP4) {                                 // reference :198-219
        const uint8_t* b = blk<T>(row + (int64_t)u * 17);
        for (int i = 0; i < 32; ++i) v[i] = mxfp4_value(b[0], nib32(b + 1, i));
    } else if constexpr (T == T_NVFP4) {                                 // reference :230-236
        // half h of the 64-value block: sub-blocks 2h, 2h + 1 of 16 (scale byte s; codes: the low nibbles of bytes
        // 4 + 8s .. 11 + 8s, then their high nibbles)
        const uint8_t* b = blk<T>(row + (int64_t)(u >> 1) * 36);
        const int h = u & 1;
        for (int i = 0; i < 32; ++i) {
            const int s = 2 * h + (i >> 4), ii = i & 15;
            const uint32_t byte = b[4 + 8 * s + (ii & 7)];
            v[i] = ue4m3_half(b[s]) * kFP4[ii < 8 ? byte & 15u : byte >> 4];
        }
    } else {
        // 256-value super-blocks: group j (values 32j .. 32j + 31) of super-block u / 8
        const int j = u & 7, hh = j >> 2, si = j & 3;
        if constexpr (T == T_Q2_K) {                                     // reference :106-114
            const uint8_t* b = blk<T>(row + (int64_t)(u >> 3) * 84);
            const float d = f16f(le16(b + 80)), dmin = f16f(le16(b + 82));
            for (int half = 0; half < 2; ++half) {                       // sub-block 2j + half of 16 values
                const uint32_t s = b[2 * j + half];
                const float dl = d * (float)(s & 15u), ml = dmin * (float)(s >> 4);
                for (int l = 0; l < 16; ++l) {
                    const int i = 16 * half + l;
                    v[i] = dl * (float)((b[16 + 32 * hh + i] >> (2 * si)) & 3u) - ml;
                }
            }
        } else if constexpr (T == T_Q3_K) {                              // reference :117-129
            const uint8_t* b = blk<T>(row + (int64_t)(u >> 3) * 110);
            const float d = f16f(le16(b + 108));
            for (int half = 0; half < 2; ++half) {
                const int sb = 2 * j + half;                             // scale: low 4 bits from bytes 96-103, high 2 from 104-107
                const uint32_t lo = sb < 8 ? (b[96 + sb] & 15u) : (b[96 + sb - 8] >> 4);
                const uint32_t hi = (b[104 + (sb & 3)] >> (2 * (sb >> 2))) & 3u;
                const float dl = d * (float)((int)(lo | (hi << 4)) - 32);
                for (int l = 0; l < 16; ++l) {
                    const int i = 16 * half + l;
                    const int q = (int)((b[32 + 32 * hh + i] >> (2 * si)) & 3u) - (((b[i] >> j) & 1u) ? 0 : 4);
                    v[i] = dl * (float)q;
                }
            }
        } else if constexpr (T == T_IQ4_XS) {                            // reference :359-369
            const uint8_t* b = blk<T>(row + (int64_t)(u >> 3) * 136);
            const uint32_t lo = (b[4 + (j >> 1)] >> (4 * (j & 1))) & 15u, hi = (le16(b + 2) >> (2 * j)) & 3u;
            const float dl = f16f(le16(b)) * (float)((int)(lo | (hi << 4)) - 32);
            for (int i = 0; i < 32; ++i) v[i] = dl * kIQ4[nib32(b + 8 + 16 * j, i)];
        } else if constexpr (T == T_TQ1_0) {                             // reference :176-185
            const uint8_t* b = blk<T>(row + (int64_t)(u >> 3) * 54);
            const float d = f16f(le16(b + 52));
            for (int i = 0; i < 32; ++i) v[i] = d * (float)tq1_code(b, 32 * j + i);
        } else {                                                         // TQ2_0, reference :188-192
            static_assert(T == T_TQ2_0, "a raw type");
            const uint8_t* b = blk<T>(row + (int64_t)(u >> 3) * 66);
            const float d = f16f(le16(b + 64));
            for (int i = 0; i < 32; ++i) v[i] = d * (float)((int)((b[32 * hh + i] >> (2 * si)) & 3u) - 1);
        }
    }
}

// bytes of one row of K values in the file's blocks of type T
template <int T>
__host__ __device__ constexpr int64_t raw_row_bytes(int64_t K) {
    return T == T_F32 ? 4 * K : (T == T_F16 || T == T_BF16) ? 2 * K : T == T_Q4_1 ? K / 32 * 20 : T == T_Q5_0 ? K / 32 * 22
         : T == T_Q5_1 ? K / 32 * 24 : T == T_IQ4_NL ? K / 32 * 18 : T == T_MXFP4 ? K / 32 * 17 : T == T_NVFP4 ? K / 64 * 36
         : T == T_Q2_K ? K / 256 * 84 : T == T_Q3_K ? K / 256 * 110 : T == T_IQ4_XS ? K / 256 * 136
         : T == T_TQ1_0 ? K / 256 * 54 : K / 256 * 66;
}


// ------------------------------------------------------------------------------------------- a unit, loaded wide
// raw_unit again, in two halves for the kernels that stream units: RawRegs holds unit u's bytes as raw_load brings them
// in (16-byte loads at any byte alignment, every byte inside the unit's own block), raw_scales its block scales, and
// raw_vals<T>(.., s, v) values 8s .. 8s + 7, the same float32 bits as raw_unit: a code byte converted exactly, then one
// product, or for the types with a minimum one FMA whose product is exact (Q4_1, Q5_1: d q + m; Q2_K: dl q - ml).
// Byte reads of these 17- to 210-byte blocks cost up to 70 load instructions a unit; these take 2 to 5.
typedef u32x4 __attribute__((aligned(1))) u32x4_u;
typedef u32x2 __attribute__((aligned(1))) u32x2_u;
typedef uint32_t __attribute__((aligned(1))) u32_u;
typedef uint16_t __attribute__((aligned(1))) u16_u;

// dwords of a unit's registers (TQ1_0, whose base-3 digits lie scattered, holds its 32 values)
template <int T>
__host__ __device__ constexpr int raw_words() {
    return T == T_F32 || T == T_TQ1_0 ? 32 : T == T_F16 || T == T_BF16 ? 16 : T == T_Q3_K ? 20 : T == T_Q2_K ? 10
         : T == T_TQ2_0 ? 9 : T == T_Q5_0 || T == T_Q5_1 || T == T_IQ4_XS ? 6 : 5;
}
// bfloat16 terms that hold every weight value of type T exactly: a value of at most 8 significant bits is one (MXFP4: 2
// bits; NVFP4: a 4-bit scale times 2 bits), of at most 16 two (F16: 11; Q5_0: an 11-bit scale times 5 bits; TQ1_0,
// TQ2_0: 11), any float32 three
template <int T>
__host__ __device__ constexpr int raw_terms() {
    return T == T_BF16 || T == T_MXFP4 || T == T_NVFP4 ? 1 : T == T_F16 || T == T_Q5_0 || T == T_TQ1_0 || T == T_TQ2_0 ? 2 : 3;
}
template <int T> struct RawRegs { uint32_t w[raw_words<T>()]; };
struct RawScales { float s[2], b[2]; };              // of values 0-15 and 16-31: scale and (types with a minimum) offset

template <int T>
__device__ __forceinline__ void raw_get16(RawRegs<T>& r, int at, const uint8_t* p) {
    const u32x4 v = *reinterpret_cast<const u32x4_u*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) r.w[at + i] = v[i];
}
template <int T>
__device__ __forceinline__ void raw_get8(RawRegs<T>& r, int at, const uint8_t* p) {
    const u32x2 v = *reinterpret_cast<const u32x2_u*>(p);
    r.w[at] = v[0];
    r.w[at + 1] = v[1];
}

template <int T>
__device__ __forceinline__ void raw_load(RawRegs<T>& r, const uint8_t* __restrict__ row, int u) {
    if constexpr (T == T_F32 || T == T_F16 || T == T_BF16) {
        constexpr int NB = T == T_F32 ? 128 : 64;
#pragma unroll
        for (int i = 0; i < NB / 16; ++i) raw_get16<T>(r, 4 * i, row + (int64_t)u * NB + 16 * i);
    } else if constexpr (T == T_Q4_1) {
        const uint8_t* b = row + (int64_t)u * 20;
        raw_get16<T>(r, 0, b + 4);
        r.w[4] = *reinterpret_cast<const u32_u*>(b);
    } else if constexpr (T == T_Q5_0) {                   // d, the high bits and two bytes of qs
        const uint8_t* b = row + (int64_t)u * 22;
        raw_get16<T>(r, 0, b + 6);
        raw_get8<T>(r, 4, b);
    } else if constexpr (T == T_Q5_1) {
        const uint8_t* b = row + (int64_t)u * 24;
        raw_get16<T>(r, 0, b + 8);
        raw_get8<T>(r, 4, b);
    } else if constexpr (T == T_IQ4_NL) {
        const uint8_t* b = row + (int64_t)u * 18;
        raw_get16<T>(r, 0, b + 2);
        r.w[4] = *reinterpret_cast<const u16_u*>(b);
    } else if constexpr (T == T_MXFP4) {
        const uint8_t* b = row + (int64_t)u * 17;
        raw_get16<T>(r, 0, b + 1);
        r.w[4] = b[0];
    } else if constexpr (T == T_NVFP4) {
        const uint8_t* b = row + (int64_t)(u >> 1) * 36;
        raw_get16<T>(r, 0, b + 4 + 16 * (u & 1));
        r.w[4] = *reinterpret_cast<const u16_u*>(b + 2 * (u & 1));
    } else if constexpr (T == T_Q2_K) {
        const uint8_t* b = row + (int64_t)(u >> 3) * 84;
        const int j = u & 7;
        raw_get16<T>(r, 0, b + 16 + 32 * (j >> 2));
        raw_get16<T>(r, 4, b + 32 + 32 * (j >> 2));
        r.w[8] = *reinterpret_cast<const u32_u*>(b + 80);
        r.w[9] = *reinterpret_cast<const u16_u*>(b + 2 * j);
    } else if constexpr (T == T_Q3_K) {                   // the last load: bytes 94-109, the 12 scale bytes and d among them
        const uint8_t* b = row + (int64_t)(u >> 3) * 110;
        const int j = u & 7;
        raw_get16<T>(r, 0, b + 32 + 32 * (j >> 2));
        raw_get16<T>(r, 4, b + 48 + 32 * (j >> 2));
        raw_get16<T>(r, 8, b);
        raw_get16<T>(r, 12, b + 16);
        raw_get16<T>(r, 16, b + 94);
    } else if constexpr (T == T_IQ4_XS) {
        const uint8_t* b = row + (int64_t)(u >> 3) * 136;
        raw_get16<T>(r, 0, b + 8 + 16 * (u & 7));
        raw_get8<T>(r, 4, b);
    } else if constexpr (T == T_TQ2_0) {
        const uint8_t* b = row + (int64_t)(u >> 3) * 66;
        const int j = u & 7;
        raw_get16<T>(r, 0, b + 32 * (j >> 2));
        raw_get16<T>(r, 4, b + 16 + 32 * (j >> 2));
        r.w[8] = *reinterpret_cast<const u16_u*>(b + 64);
    } else {
        static_assert(T == T_TQ1_0, "a raw type");
        float v[32];
        raw_unit<T>(row, u, v);
#pragma unroll
        for (int i = 0; i < 32; ++i) r.w[i] = __float_as_uint(v[i]);
    }
}

template <int T>
__device__ __forceinline__ RawScales raw_scales(const RawRegs<T>& r, int u) {
    RawScales o{};
    const int j = u & 7;
    if constexpr (T == T_Q4_1 || T == T_Q5_1) {
        o.s[0] = o.s[1] = f16f(r.w[4]);
        o.b[0] = o.b[1] = f16f(r.w[4] >> 16);
    } else if constexpr (T == T_Q5_0 || T == T_IQ4_NL) {
        o.s[0] = o.s[1] = f16f(r.w[4]);
    } else if constexpr (T == T_MXFP4) {                  // 2^(e - 128); e = 0, 1: the subnormals 2^-128, 2^-127
        const uint32_t e = r.w[4];
        o.s[0] = o.s[1] = __uint_as_float(e >= 2u ? (e - 1u) << 23 : 0x00200000u << e);
    } else if constexpr (T == T_NVFP4) {
        o.s[0] = ue4m3_half(r.w[4] & 0xFFu);
        o.s[1] = ue4m3_half(r.w[4] >> 8);
    } else if constexpr (T == T_Q2_K) {
        const float d = f16f(r.w[8]), dmin = f16f(r.w[8] >> 16);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t c = (r.w[9] >> (8 * h)) & 0xFFu;
            o.s[h] = d * (float)(c & 15u);
            o.b[h] = -(dmin * (float)(c >> 4));
        }
    } else if constexpr (T == T_Q3_K) {
        const uint32_t s0 = __builtin_amdgcn_alignbit(r.w[17], r.w[16], 16), s1 = __builtin_amdgcn_alignbit(r.w[18], r.w[17], 16);
        const uint32_t s2 = __builtin_amdgcn_alignbit(r.w[19], r.w[18], 16);
        const uint32_t lo = ((j & 2) ? s1 : s0) >> (16 * (j & 1) + 4 * (j >> 2));
        const uint32_t hi = s2 >> (16 * (j & 1) + 2 * (j >> 1));
        const uint32_t c = (lo & 0x0F0Fu) | ((hi & 0x0303u) << 4);
        const float d = f16f(r.w[19] >> 16);
        o.s[0] = d * (float)((int)(c & 0xFFu) - 32);
        o.s[1] = d * (float)((int)(c >> 8) - 32);
    } else if constexpr (T == T_IQ4_XS) {                 // d, scales_h | scales_l
        const uint32_t lo = (r.w[5] >> (4 * j)) & 15u, hi = (r.w[4] >> (16 + 2 * j)) & 3u;
        o.s[0] = o.s[1] = f16f(r.w[4]) * (float)((int)(lo | (hi << 4)) - 32);
    } else if constexpr (T == T_TQ2_0) {
        o.s[0] = o.s[1] = f16f(r.w[8]);
    } else if constexpr (T == T_BF16) {
        o.s[0] = o.s[1] = 1.f;
    }
    return o;
}

// the signed bytes of a 16-entry table (t: entries 0-3, 4-7, 8-11, 12-15) at the 4 nibbles of n (one a byte)
__device__ __forceinline__ uint32_t nib_lookup(uint32_t n, const uint32_t t[4]) {
    const uint32_t i = n & 0x07070707u;
    const uint32_t a = __builtin_amdgcn_perm(t[1], t[0], i), b = __builtin_amdgcn_perm(t[3], t[2], i);
    return __builtin_amdgcn_perm(b, a, ((n >> 1) & 0x04040404u) | 0x03020100u);
}
// bits 0-3 of x as bit 0 of the four bytes
__device__ __forceinline__ uint32_t spread4(uint32_t x) { return (__umul24(x & 15u, 0x00204081u)) & 0x01010101u; }

template <int T>
__device__ __forceinline__ void raw_vals(const RawRegs<T>& r, const RawScales& sc, int u, int s, float v[8]) {
    const int j = u & 7;
    if constexpr (T == T_F32 || T == T_TQ1_0) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = __uint_as_float(r.w[8 * s + e]);
    } else if constexpr (T == T_F16 || T == T_BF16) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t w = r.w[4 * s + (e >> 1)];
            if constexpr (T == T_BF16) v[e] = __uint_as_float((e & 1) ? w & 0xFFFF0000u : w << 16);
            else v[e] = f16f((e & 1) ? w >> 16 : w);
        }
    } else {
        constexpr bool MIN = T == T_Q4_1 || T == T_Q5_1 || T == T_Q2_K;
        uint32_t c[2];                                    // the codes of values 8s .. 8s + 3 and 8s + 4 .. 8s + 7, a byte each
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if constexpr (T == T_Q2_K || T == T_Q3_K || T == T_TQ2_0) {
                c[h] = (r.w[2 * s + h] >> (2 * (j & 3))) & 0x03030303u;
                if constexpr (T == T_Q3_K) c[h] |= ((r.w[8 + 2 * s + h] >> j) & 0x01010101u) << 2;
                if constexpr (T == T_Q3_K) c[h] = (c[h] + 0x7C7C7C7Cu) ^ 0x80808080u;            // - 4
                if constexpr (T == T_TQ2_0) c[h] = (c[h] + 0x7F7F7F7Fu) ^ 0x80808080u;           // - 1
            } else if constexpr (T == T_NVFP4) {          // sub-block s / 2 of 16: low nibbles of its 8 bytes, then the high ones
                c[h] = (r.w[2 * (s >> 1) + h] >> (4 * (s & 1))) & 0x0F0F0F0Fu;
            } else {                                      // 16 bytes: low nibbles, then the high ones
                c[h] = (r.w[2 * (s & 1) + h] >> (4 * (s >> 1))) & 0x0F0F0F0Fu;
            }
            if constexpr (T == T_Q5_0 || T == T_Q5_1) {
                const uint32_t qh = T == T_Q5_1 ? r.w[5] : __builtin_amdgcn_alignbit(r.w[5], r.w[4], 16);
                c[h] |= spread4(qh >> (8 * s + 4 * h)) << 4;
                if constexpr (T == T_Q5_0) c[h] = (c[h] + 0x70707070u) ^ 0x80808080u;            // - 16
            }
            if constexpr (T == T_IQ4_NL || T == T_IQ4_XS) {                                      // kIQ4
                const uint32_t t[4] = {0xBFAD9881u, 0xF6EADDCFu, 0x26190D01u, 0x71594535u};
                c[h] = nib_lookup(c[h], t);
            }
            if constexpr (T == T_MXFP4 || T == T_NVFP4) {                                        // kFP4
                const uint32_t t[4] = {0x03020100u, 0x0C080604u, 0xFDFEFF00u, 0xF4F8FAFCu};
                c[h] = nib_lookup(c[h], t);
            }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t b = c[e >> 2] >> (8 * (e & 3));
            if constexpr (MIN) v[e] = __builtin_fmaf(sc.s[s >> 1], (float)(b & 0xFFu), sc.b[s >> 1]);
            else v[e] = sc.s[s >> 1] * (float)(int8_t)b;
        }
    }
}

// ------------------------------------------------------------------------------- codes as bfloat16 pairs
// For the types whose value is scale * code (+ offset) with an integer code of at most 8 significant bits: the codes of
// values 8s .. 8s + 7 as four bfloat16 pairs, exact, so that a unit's products with x sum unscaled (v_dot2_f32_bf16) and the
// scale multiplies the sum of 16 or 32. BF16's values are their own codes (scale 1). Codes of up to 16 values come from byte
// tables of their bfloat16 halves (a byte permute per 4 codes each), the others through a float32 conversion.
template <int T>
__host__ __device__ constexpr bool raw_coded() { return T != T_F32 && T != T_F16 && T != T_TQ1_0; }
template <int T>
__host__ __device__ constexpr bool raw_min() { return T == T_Q4_1 || T == T_Q5_1 || T == T_Q2_K; }

// bfloat16 bits of a small integer; entries 4i .. 4i + 3 of a table of them: their low (b = 0) or high (1) bytes
__host__ __device__ constexpr uint32_t bf16_int(int v) {
    uint32_t m = (uint32_t)(v < 0 ? -v : v), e = 0;
    if (m == 0) return 0;
    while (m >> (e + 1)) ++e;
    return (v < 0 ? 0x8000u : 0u) | ((127u + e) << 7) | ((e <= 7 ? m << (7 - e) : m >> (e - 7)) & 0x7Fu);
}
struct CodeTable { uint32_t b[2][4]; };
template <int N>
__host__ __device__ constexpr CodeTable code_table(const int (&v)[N]) {
    CodeTable t{};
    for (int i = 0; i < N; ++i)
        for (int h = 0; h < 2; ++h) t.b[h][i >> 2] |= ((bf16_int(v[i]) >> (8 * h)) & 0xFFu) << (8 * (i & 3));
    return t;
}
template <int T>
__host__ __device__ constexpr CodeTable raw_table() {
    constexpr int q2[4] = {0, 1, 2, 3}, q3[8] = {-4, -3, -2, -1, 0, 1, 2, 3}, tq[4] = {-1, 0, 1, 2};
    constexpr int iq[16] = {-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113};
    constexpr int fp[16] = {0, 1, 2, 3, 4, 6, 8, 12, 0, -1, -2, -3, -4, -6, -8, -12};
    constexpr int q4[16] = {0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15};
    return T == T_Q2_K ? code_table(q2) : T == T_Q3_K ? code_table(q3) : T == T_TQ2_0 ? code_table(tq)
         : T == T_Q4_1 ? code_table(q4) : T == T_MXFP4 || T == T_NVFP4 ? code_table(fp) : code_table(iq);
}

template <int T>
__device__ __forceinline__ void raw_pairs(const RawRegs<T>& r, int u, int s, uint32_t p[4]) {
    static_assert(raw_coded<T>(), "a type of codes");
    const int j = u & 7;
    if constexpr (T == T_BF16) {
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = r.w[4 * s + i];
    } else {
#pragma unroll
        for (int h = 0; h < 2; ++h) {                     // values 8s + 4h .. + 3
            uint32_t lo, hi;
            if constexpr (T == T_Q2_K || T == T_Q3_K || T == T_TQ2_0) {
                constexpr CodeTable t = raw_table<T>();
                uint32_t c = (r.w[2 * s + h] >> (2 * (j & 3))) & 0x03030303u;
                if constexpr (T == T_Q3_K) c |= ((r.w[8 + 2 * s + h] >> j) & 0x01010101u) << 2;
                lo = __builtin_amdgcn_perm(t.b[0][1], t.b[0][0], c);
                hi = __builtin_amdgcn_perm(t.b[1][1], t.b[1][0], c);
            } else if constexpr (T == T_Q5_0 || T == T_Q5_1) {
                uint32_t c = (r.w[2 * (s & 1) + h] >> (4 * (s >> 1))) & 0x0F0F0F0Fu;
                const uint32_t qh = T == T_Q5_1 ? r.w[5] : __builtin_amdgcn_alignbit(r.w[5], r.w[4], 16);
                c |= spread4(qh >> (8 * s + 4 * h)) << 4;
                if constexpr (T == T_Q5_0) c = (c + 0x70707070u) ^ 0x80808080u;
                p[2 * h] = T == T_Q5_0 ? i8_pair(c, 0) : u8_pair(c, 0);
                p[2 * h + 1] = T == T_Q5_0 ? i8_pair(c, 1) : u8_pair(c, 1);
                continue;
            } else {
                constexpr CodeTable t = raw_table<T>();
                const uint32_t c = T == T_NVFP4 ? (r.w[2 * (s >> 1) + h] >> (4 * (s & 1))) & 0x0F0F0F0Fu
                                                : (r.w[2 * (s & 1) + h] >> (4 * (s >> 1))) & 0x0F0F0F0Fu;
                const uint32_t i = c & 0x07070707u, sel = ((c >> 1) & 0x04040404u) | 0x03020100u;
                lo = __builtin_amdgcn_perm(__builtin_amdgcn_perm(t.b[0][3], t.b[0][2], i), __builtin_amdgcn_perm(t.b[0][1], t.b[0][0], i), sel);
                hi = __builtin_amdgcn_perm(__builtin_amdgcn_perm(t.b[1][3], t.b[1][2], i), __builtin_amdgcn_perm(t.b[1][1], t.b[1][0], i), sel);
            }
            p[2 * h] = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
            p[2 * h + 1] = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
        }
    }
}

// whether a unit's values, where their scales are finite, are finite themselves (MXFP4's largest scales overflow: 12 * 2^125)
template <int T>
__device__ __forceinline__ bool raw_finite(const RawScales& sc) {
    if constexpr (T == T_MXFP4) return sc.s[0] <= 0x1p124f;
    else return true;
}

// ------------------------------------------------------------------------- a super-block, shared by 8 lanes
// The 2- and 3-bit types' super-blocks, whose bytes several of their 8 units share: 8 lanes load one with a 16-byte load
// each (raw_part: the block's 16-byte pieces, the last one ending with the block) and leave it in LDS, RAW_SLOT bytes a
// super-block (the padding spreads 8 of them over the banks), from where each lane takes its unit's registers (raw_take).
template <int T>
__host__ __device__ constexpr bool raw_shared() { return T == T_Q2_K || T == T_Q3_K || T == T_TQ2_0; }
constexpr int RAW_SLOT = 144;
template <int T>
__device__ __forceinline__ u32x4 raw_part(const uint8_t* __restrict__ row, int sb, int j) {
    constexpr int NB = T == T_Q2_K ? 84 : T == T_Q3_K ? 110 : 66;
    return *reinterpret_cast<const u32x4_u*>(row + (int64_t)sb * NB + (16 * j < NB - 16 ? 16 * j : NB - 16));
}
template <int T>
__device__ __forceinline__ void raw_take(RawRegs<T>& r, const uint8_t* slot, int j) {
    constexpr int NB = T == T_Q2_K ? 84 : T == T_Q3_K ? 110 : 66, LAST = (NB - 1) / 16 * 16;   // the last piece's place
    constexpr int Q = T == T_Q2_K ? 16 : T == T_Q3_K ? 32 : 0;
    const u32x4 a = ld16(slot + Q + 32 * (j >> 2)), b = ld16(slot + Q + 16 + 32 * (j >> 2));
#pragma unroll
    for (int i = 0; i < 4; ++i) r.w[i] = a[i], r.w[4 + i] = b[i];
    if constexpr (T == T_Q3_K) {
        const u32x4 c = ld16(slot), d = ld16(slot + 16), e = ld16(slot + LAST);
#pragma unroll
        for (int i = 0; i < 4; ++i) r.w[8 + i] = c[i], r.w[12 + i] = d[i], r.w[16 + i] = e[i];
    } else if constexpr (T == T_Q2_K) {
        r.w[8] = *reinterpret_cast<const uint32_t*>(slot + LAST + 12);
        r.w[9] = *reinterpret_cast<const uint16_t*>(slot + 2 * j);
    } else {
        r.w[8] = *reinterpret_cast<const uint32_t*>(slot + LAST + 12) >> 16;
    }
}

}  // namespace mbq
