// gfx950 kernels of the exact path's fused products: y (M, N) = x (M, K) @ W.T straight from the file's blocks of the
// ggml types without kernel planes, each weight value rebuilt in registers (mbq_raw_unit.h: bit for bit the values
// mbq_dequant_raw writes) instead of written as float32 and read back. Reference src/mashbox/ops/__init__.py:574-576,
// 624-632 (dequant, then a float32 dot).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <type_traits>

#include "mbq_device.h"
#include "mbq_launch.h"
#include "mbq_layout.h"
#include "mbq_raw_unit.h"

namespace mbq {

static int check_launch(const char* what) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(MBQ_LAUNCH_FAIL, "%s: %s", what, hipGetErrorString(e));
    return 0;
}

// 8 values -> NT bfloat16 operands whose sum they are
template <int NT>
__device__ __forceinline__ void raw_split(const float v[8], bf16x8_t b[NT]) {
#pragma clang fp contract(off)                                          // v's own bits: not the product behind them, unrounded
    uint32_t t[NT][4];
    float f[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = v[e];
#pragma unroll
    for (int k = 0; k < NT; ++k) {
#pragma unroll
        for (int e = 0; e < 8; e += 2) t[k][e >> 1] = __builtin_amdgcn_perm(__float_as_uint(f[e + 1]), __float_as_uint(f[e]), 0x07060302u);
        if (k + 1 < NT)
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] -= __uint_as_float(__float_as_uint(f[e]) & 0xFFFF0000u);
        b[k] = __builtin_bit_cast(bf16x8_t, u32x4{t[k][0], t[k][1], t[k][2], t[k][3]});
    }
}

// ------------------------------------------------------------------------------------------------ 1-8 rows
// Each lane takes one 32-value unit at a time and multiplies it with up to MR activation rows: the types of codes
// (raw_coded) as bfloat16 pairs with v_dot2_f32_bf16, float32 sums of exact products that the scale multiplies once (a unit
// that meets a scale, an activation or a sum that is not finite: value by value); F16 at 5-8 rows as two
// bfloat16 terms per value (1024 x 5120 at 8 rows 13.5 us value by value, 10.9 so); F32, TQ1_0 and F16 at 1-4 rows value by
// value with float32 FMAs (F16 34816 x 5120 at 4 rows 68 us, 77 as two terms). A unit's sum is added to the row's. Bound: the vector work (2.5 to 4 instructions per value at one row) and, below about 20 MB, the
// launch's fill and drain. Against a float64 product it is off by 0.6e-7 to 1.5e-7 (one to eight rows, K 512 to 17408).
//
// 8 lanes take 8 consecutive units of a weight row (a super-block of the 256-value types: lane j always its sub-block j, so
// the shifts of its codes and scales are the lane's constants), a wave 8 rows. The RV_W waves of a block take the 8-unit
// steps of the same rows in turn (KS of them) or other rows. x is staged once per block in LDS as it comes, RV_X1 or RV_X
// bytes at a time, a super-block's 16-byte pieces in the order [piece][unit], which the 8 lanes read as 128 consecutive
// bytes. The bytes of the next step are in flight while a step computes.
//
// One row, us (before: 16 to 64 lanes per row, the blocks read a byte or a dword at a time): Q3_K 34816 x 5120 82 -> 27,
// 5120 x 17408 56 -> 17, 8192 x 5120 24 -> 9.6; IQ4_XS 112 -> 29, 60 -> 18; Q5_0 59 -> 35, 28 -> 21; F16 63 -> 60. Four
// rows: Q3_K 34816 x 5120 128 -> 43. Two rows of weights per lane (half the LDS reads of x) ran 2 % faster on 34816 rows and
// 10-20 % slower below 8192, 4 waves per block 5-15 % slower at 5120 x 17408: neither is kept.
constexpr int RV_W = 8, RV_X1 = 40 * 1024, RV_X = 64 * 1024, RV_XL = 128 * 1024;

// a step's bytes in flight: a 16-byte piece of a super-block (raw_shared), else the unit itself
template <int T, bool SH = raw_shared<T>()> struct RawFlight { RawRegs<T> u; };
template <int T> struct RawFlight<T, true> { u32x4 p; };

template <int T, int MR>
__global__ __launch_bounds__(64 * RV_W) void raw_gemv_kernel(const uint8_t* __restrict__ raw, const uint16_t* __restrict__ x, int M,
                                                             int N, int K, void* __restrict__ y, int out_bf16, int KS, int KC) {
    constexpr bool SH = raw_shared<T>();
    extern __shared__ __align__(16) uint16_t xs[];                       // [M][KC], the waves' sums, their super-blocks
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, j = lane & 7;
    const int U = K >> 5, ks = wave % KS, RB = RV_W / KS * 8;            // RB: rows of the block
    const int n = blockIdx.x * RB + wave / KS * 8 + (lane >> 3);
    float* const red = reinterpret_cast<float*>(xs + M * KC);            // [wave][8 rows][MR]
    uint8_t* const sb = reinterpret_cast<uint8_t*>(red + RV_W * 8 * MR) + (wave * 8 + (lane >> 3)) * RAW_SLOT;
    const uint8_t* row = raw + (int64_t)(n < N ? n : N - 1) * raw_row_bytes<T>(K);
    float acc[MR];
#pragma unroll
    for (int m = 0; m < MR; ++m) acc[m] = 0.f;

    for (int c0 = 0; c0 < K; c0 += KC) {
        const int kc = K - c0 < KC ? K - c0 : KC, steps = (kc + 255) >> 8, u0 = c0 >> 5;
        RawFlight<T> fl;
        auto load = [&](int i) {                                         // past the end: the last unit again
            const int u = u0 + 8 * (i < steps ? i : steps - 1) + j;
            if constexpr (SH) fl.p = raw_part<T>(row, u >> 3, j);
            else raw_load<T>(fl.u, row, u < U ? u : U - 1);
        };
        load(ks);
        if (c0) {                                                        // the last chunk's x has been read
            wait_lgkm0();                                                // (and no LDS write of the wave is in flight)
            __syncthreads();
        }
        for (int q = threadIdx.x; q < M * (kc >> 3); q += 64 * RV_W) {
            const int m = q / (kc >> 3), p = q % (kc >> 3);              // piece p: unit p / 4, its piece p % 4
            st16(xs + m * KC + (p >> 5) * 256 + ((p & 3) * 8 + ((p >> 2) & 7)) * 8, ld16(x + (int64_t)m * K + c0 + 8 * p));
        }
        __syncthreads();
        for (int i = ks; i < steps; i += KS) {
            RawRegs<T> cur;
            if constexpr (SH) {
                st16(sb + 16 * j, fl.p);
                __builtin_amdgcn_wave_barrier();                         // a wave's LDS accesses complete in order
                raw_take<T>(cur, sb, j);
                __builtin_amdgcn_wave_barrier();
            } else {
                cur = fl.u;
            }
            load(i + KS);
            const int u = u0 + 8 * i + j;
            if (u >= U) continue;
            const RawScales sc = raw_scales<T>(cur, u);
            const uint16_t* xp = xs + i * 256 + j * 8;
            float d[MR];                                                 // the unit's sums
#pragma unroll
            for (int m = 0; m < MR; ++m) d[m] = 0.f;
            bool done = false;
            if constexpr (raw_coded<T>()) {
                constexpr int HV = T == T_Q2_K || T == T_Q3_K || T == T_NVFP4 ? 2 : 1;       // scales of a unit
#pragma unroll
                for (int h = 0; h < HV; ++h) {
                    float t[MR], sx[MR];
#pragma unroll
                    for (int m = 0; m < MR; ++m) t[m] = sx[m] = 0.f;
#pragma unroll
                    for (int s = h * (4 / HV); s < (h + 1) * (4 / HV); ++s) {
                        uint32_t p[4];
                        raw_pairs<T>(cur, u, s, p);
#pragma unroll
                        for (int m = 0; m < MR; ++m) {
                            if (MR > 1 && m >= M) break;
                            const u32x4 q = ld16(xp + m * KC + s * 64);
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                if constexpr (raw_min<T>()) sx[m] = dot2(BF16_ONES, q[e], sx[m]);
                                t[m] = dot2(p[e], q[e], t[m]);
                            }
                        }
                    }
#pragma unroll
                    for (int m = 0; m < MR; ++m) {
                        d[m] = __builtin_fmaf(sc.s[h], t[m], d[m]);
                        if constexpr (raw_min<T>()) d[m] = __builtin_fmaf(sc.b[h], sx[m], d[m]);
                    }
                }
                done = raw_finite<T>(sc);
            } else if constexpr (T == T_F16 && MR == 8) {                // two exact terms: a dot2 each for two values
                done = true;
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    float v[8];
                    bf16x8_t b[2];
                    raw_vals<T>(cur, sc, u, s, v);
                    raw_split<2>(v, b);
                    const u32x4 hi = __builtin_bit_cast(u32x4, b[0]), lo = __builtin_bit_cast(u32x4, b[1]);
#pragma unroll
                    for (int m = 0; m < MR; ++m) {
                        if (m >= M) break;
                        const u32x4 q = ld16(xp + m * KC + s * 64);
#pragma unroll
                        for (int e = 0; e < 4; ++e) d[m] = dot2(lo[e], q[e], dot2(hi[e], q[e], d[m]));
                    }
                }
            }
            if (done) {
                float f = 0.f;                                           // a non-finite scale, activation or sum makes it NaN
#pragma unroll
                for (int m = 0; m < MR; ++m) f = __builtin_fmaf(0.f, d[m], f);
                done = f == 0.f;
            }
            if (!done) {
#pragma unroll
                for (int m = 0; m < MR; ++m) d[m] = 0.f;
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    float v[8];
                    raw_vals<T>(cur, sc, u, s, v);
#pragma unroll
                    for (int m = 0; m < MR; ++m) {
                        if (MR > 1 && m >= M) break;
                        const u32x4 q = ld16(xp + m * KC + s * 64);
#pragma unroll
                        for (int e = 0; e < 8; ++e)
                            d[m] = __builtin_fmaf(__uint_as_float((e & 1) ? q[e >> 1] & 0xFFFF0000u : q[e >> 1] << 16), v[e], d[m]);
                    }
                }
            }
#pragma unroll
            for (int m = 0; m < MR; ++m) acc[m] += d[m];
        }
    }
#pragma unroll
    for (int m = 0; m < MR; ++m) {
        float t = acc[m];
        t += dpp_f<0xB1, 0xF>(t);                                        // quad_perm [1,0,3,2]
        t += dpp_f<0x4E, 0xF>(t);                                        // quad_perm [2,3,0,1]
        t += dpp_f<0x141, 0xF>(t);                                       // row_half_mirror: the other quad of the 8 lanes
        if (j == 0) red[(wave * 8 + (lane >> 3)) * MR + m] = t;
    }
    __syncthreads();
    for (int q = threadIdx.x; q < RB * M; q += 64 * RV_W) {              // the block's rows in order, a row's KS sums in order
        const int rr = q % RB, m = q / RB, no = blockIdx.x * RB + rr;
        if (no >= N) continue;
        const float* p = red + (rr / 8 * KS * 8 + rr % 8) * MR + m;
        float t = p[0];
        for (int k = 1; k < KS; ++k) t += p[k * 8 * MR];
        store_y(y, (int64_t)m * N + no, t, out_bf16);
    }
}

// Waves per row: 4, or 8 below 8192 rows, where 4 leave CUs idle (one row, 4 against 8: Q3_K 5120 x 17408 21.5 / 17.0 us,
// 5120 x 6144 9.6 / 8.4; 34816 x 5120 26.9 / 28.2, 9728 x 2560 7.7 / 7.9); never more than a row has 8-unit steps
template <int T, int MR>
static int raw_gemv_m(const uint8_t* raw, const uint16_t* x, int64_t M, int64_t N, int64_t K, void* y, int out_bf16, hipStream_t s) {
    int KS = N < 8192 ? 8 : 4;
    while (KS > 1 && KS * 256 > K) KS /= 2;
    const int64_t rows = RV_W / KS * 8, blocks = (N + rows - 1) / rows;
    const int64_t X = M == 1 ? RV_X1 : blocks <= cus_of_device() ? RV_XL : RV_X;
    const int64_t KC = std::min<int64_t>((K + 255) / 256 * 256, X / (2 * M) / 256 * 256);
    const size_t lds = (size_t)(M * KC) * 2 + (size_t)RV_W * 8 * (MR * 4 + (raw_shared<T>() ? RAW_SLOT : 0));
    auto kern = raw_gemv_kernel<T, MR>;
    static std::atomic<uint64_t> set{0};
    if (set_lds_limit((const void*)kern, RV_XL + 16 * 1024, set) != hipSuccess) return set_error(MBQ_LAUNCH_FAIL, "raw GEMV: %zu bytes of LDS refused", lds);
    kern<<<dim3((unsigned)blocks), 64 * RV_W, lds, s>>>(raw, x, (int)M, (int)N, (int)K, y, out_bf16, KS, (int)KC);
    return check_launch("raw GEMV");
}

template <int T>
static int raw_gemv_t(const uint8_t* raw, const uint16_t* x, int64_t M, int64_t N, int64_t K, void* y, int out_bf16, hipStream_t s) {
    if (M == 1) return raw_gemv_m<T, 1>(raw, x, M, N, K, y, out_bf16, s);
    if (M == 2) return raw_gemv_m<T, 2>(raw, x, M, N, K, y, out_bf16, s);
    if (M <= 4) return raw_gemv_m<T, 4>(raw, x, M, N, K, y, out_bf16, s);
    return raw_gemv_m<T, 8>(raw, x, M, N, K, y, out_bf16, s);
}

int launch_raw_gemv(int t, const uint8_t* raw, const uint16_t* x, int64_t M, int64_t N, int64_t K, void* y, int out_bf16,
                    hipStream_t s) {
    switch (t) {
#define RAW_CASE(T) case T: return raw_gemv_t<T>(raw, x, M, N, K, y, out_bf16, s);
        RAW_CASE(T_F32) RAW_CASE(T_F16) RAW_CASE(T_BF16) RAW_CASE(T_Q4_1) RAW_CASE(T_Q5_0) RAW_CASE(T_Q5_1) RAW_CASE(T_Q2_K)
        RAW_CASE(T_Q3_K) RAW_CASE(T_IQ4_NL) RAW_CASE(T_IQ4_XS) RAW_CASE(T_TQ1_0) RAW_CASE(T_TQ2_0) RAW_CASE(T_MXFP4) RAW_CASE(T_NVFP4)
#undef RAW_CASE
    }
    return set_error(MBQ_BAD_ARG, "raw GEMV: no kernel for ggml type %d (kernel types run on their planes)", t);
}

// ------------------------------------------------------------------------------------- more rows: a bfloat16-split GEMM
// The float32 product on the bfloat16 matrix cores. x is bfloat16 as it comes; every weight value is the exact sum of
// raw_terms<T>() bfloat16 terms (its float32 bits cut into 8-bit significands: the top, then what is left, then the
// rest), so the MFMAs multiply exactly and only their float32 accumulation rounds, as a float32 GEMM's does. Against a
// float64 product (2-norm, 512 x 4096 x 5120) it is off by 1.5e-7 to 2.7e-7, the rebuild and float32 library GEMM it
// replaces by 0.7e-6 to 1.3e-6; smaller shapes alike. The float32 GEMM runs at 98 TFLOP/s here; this kernel's MFMAs at
// 1.25 PFLOP/s, 420 TFLOP/s of the product with three terms, 567 with two, 749 with one (512 rows, 34816 x 5120: Q3_K
// 434 us, F16 322, BF16 244; the rebuild and float32 GEMM 2.2 ms).
//
// Tile: 32 BMT activation rows x 256 weight rows, K step 64, 8 waves. Wave w owns weight rows 32w .. 32w + 31 and all
// the activation rows (BMT accumulators of v_mfma_f32_32x32x16_bf16): its lane l decodes unit l / 32 of the K step of row
// l % 32 straight into B operands, so no weight passes LDS and no value is decoded twice in a block; x goes through an
// LDS ring of three stages filled by DMA two steps ahead. The K values of an MFMA are the 8 of each lane half's unit
// (values 8s .. 8s + 7 of units 0 and 1 at substep s), for A and B alike. Bound: the matrix cores (BMT = 8: 96 MFMAs of
// 32 cycles per wave and step, against about 300 vector instructions of decode and split).
//
// One barrier per step. The weight bytes of the next step and the x stage after it are issued after it, weights first,
// so that at the next barrier's wait only that DMA may be outstanding: the wait counts DMA instructions alone.
//
// The tiles that do not fill a round of the CUs are cut along K into S pieces, each a block of its own, whose float32
// partials the second kernel adds in piece order. An output that is not finite (a non-finite weight or activation, whose
// lower terms are inf - inf or meet 0 * inf, or a sum past the range) is computed again value by value, so that it is what
// the float32 product gives.
constexpr int RG_T = 512, RG_BN = 256, RG_K = 64;

struct RawGemmArgs {
    const uint8_t* raw;
    const uint16_t* x;
    void* y;
    float* part;
    int M, N, K, out_bf16;
    int tm;                // tiles along M (fastest)
    int full, S, ipp;      // tiles run whole; pieces per other tile, K steps per piece
};

// one output in float32, value by value
template <int T>
__device__ __forceinline__ float raw_dot(const uint8_t* row, const uint16_t* x, int K) {
    float acc = 0.f;
    for (int u = 0; u < K / 32; ++u) {
        RawRegs<T> r;
        raw_load<T>(r, row, u);
        const RawScales sc = raw_scales<T>(r, u);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            float v[8];
            raw_vals<T>(r, sc, u, s, v);
            const u32x4 q = ld16(x + 32 * u + 8 * s);
#pragma unroll
            for (int e = 0; e < 8; ++e)
                acc = __builtin_fmaf(__uint_as_float((e & 1) ? q[e >> 1] & 0xFFFF0000u : q[e >> 1] << 16), v[e], acc);
        }
    }
    return acc;
}

// element offset of chunk c (8 values) of row r in an x stage
__device__ __forceinline__ int rg_off(int r, int c) { return r * RG_K + ((c ^ ((r >> 1) & 7)) << 3); }

// Types whose 32 values share one scale and whose codes need no more than a bfloat16's 8 bits (raw_factored): one MFMA per
// code instead of three per value. Both lane halves hold the same unit (half h its values 8h .. + 7 and 16 + 8h .. + 7, the
// low and high nibbles of bytes 8h .. + 7), so two MFMAs sum a unit alone, unscaled, and 16 FMAs per row tile add scale times
// that sum to the accumulators, behind the MFMAs of the next two row tiles. A scale that is not finite goes in as NaN. Bound:
// the FMAs and the decode, about 400 vector instructions against 32 MFMAs of 32 cycles per wave and step. IQ4_XS, 512 rows,
// against three terms: 34816 x 5120 436 -> 283 us, 5120 x 17408 220 -> 147, 8192 x 5120 115 -> 80; 16 rows 80 -> 57. Error
// against float64 2.7e-7 -> 1.0e-7. Q5_0, two terms otherwise: 512 rows 313 -> 276 us, 64 rows 78 -> 73, but
// 5120 x 6144 at 16 rows 21.4 -> 24.5, so from 33 rows.
template <int T, int BMT>
__host__ __device__ constexpr bool raw_factored() { return T == T_IQ4_NL || T == T_IQ4_XS || (T == T_Q5_0 && BMT >= 2); }
template <int T> struct RawHalf { uint32_t q[2][2], h[T == T_IQ4_XS ? 2 : 4]; };     // two units' nibbles; their headers

template <int T>
__device__ __forceinline__ void raw_half_load(RawHalf<T>& r, const uint8_t* __restrict__ row, int it, int half, int U) {
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        const int u = 2 * it + w < U ? 2 * it + w : U - 1;              // past K: the last unit again (it meets zeros)
        const uint8_t* b = row + (T == T_IQ4_XS ? (int64_t)(u >> 3) * 136 : (int64_t)u * (T == T_Q5_0 ? 22 : 18));
        const u32x2 q = *reinterpret_cast<const u32x2_u*>(b + (T == T_IQ4_XS ? 8 + 16 * (u & 7) : T == T_Q5_0 ? 6 : 2) + 8 * half);
        r.q[w][0] = q[0];
        r.q[w][1] = q[1];
        if constexpr (T == T_IQ4_NL) {
            r.h[w] = *reinterpret_cast<const u16_u*>(b);
        } else if (T == T_Q5_0 || w == 0) {
            const u32x2 h = *reinterpret_cast<const u32x2_u*>(b);
            r.h[2 * w] = h[0];
            r.h[2 * w + 1] = h[1];
        }
    }
}

// unit w's scale, and its codes as two B operands
template <int T>
__device__ __forceinline__ float raw_half_codes(const RawHalf<T>& r, int it, int w, int half, bf16x8_t b[2]) {
    RawRegs<T> g;
    g.w[0] = r.q[w][0];
    g.w[1] = r.q[w][1];
    g.w[2] = g.w[3] = 0;
    if constexpr (T == T_IQ4_NL) g.w[4] = r.h[w];
    else if constexpr (T == T_IQ4_XS) g.w[4] = r.h[0], g.w[5] = r.h[1];
    else g.w[4] = r.h[2 * w], g.w[5] = r.h[2 * w + 1];
    if constexpr (T == T_Q5_0) {                                         // the high bits of values 8h .. + 7 and 16 + 8h .. + 7
        const uint32_t qh = __builtin_amdgcn_alignbit(g.w[5], g.w[4], 16) >> (8 * half);
        g.w[5] = qh >> 16;
        g.w[4] = (g.w[4] & 0xFFFFu) | (qh << 16);
    }
    const float s = raw_scales<T>(g, 2 * it + w).s[0];
#pragma unroll
    for (int k = 0; k < 2; ++k) {                                        // raw_pairs' steps 0 and 2: low, high nibbles of w[0], w[1]
        uint32_t p[4];
        raw_pairs<T>(g, 0, 2 * k, p);
        b[k] = __builtin_bit_cast(bf16x8_t, u32x4{p[0], p[1], p[2], p[3]});
    }
    return __builtin_fabsf(s) < __builtin_inff() ? s : __builtin_nanf("");
}

template <int T, int BMT>
__global__ __launch_bounds__(RG_T, BMT >= 4 || T == T_TQ1_0 ? 2 : 4) void raw_gemm_kernel(const RawGemmArgs g) {
    constexpr int NT = raw_terms<T>(), BM = 32 * BMT, STAGE = BM * RG_K;
    constexpr bool FACT = raw_factored<T, BMT>();
    constexpr int ND = BMT >= 2 ? BMT / 2 : 1;                           // DMA instructions of a wave per stage
    extern __shared__ __align__(16) uint16_t lds[];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, col = lane & 31, half = lane >> 5;
    const int IT = (g.K + RG_K - 1) / RG_K, U = g.K >> 5;
    const int b = blockIdx.x, p = b - g.full;
    const int tile = p < 0 ? b : g.full + p / g.S;
    const int k0 = p < 0 ? 0 : (p % g.S) * g.ipp, k1 = p < 0 ? IT : (k0 + g.ipp < IT ? k0 + g.ipp : IT);
    const int m0 = (tile % g.tm) * BM, n = (tile / g.tm) * RG_BN + wave * 32 + col;
    const uint8_t* row = g.raw + (int64_t)(n < g.N ? n : g.N - 1) * raw_row_bytes<T>(g.K);

    // x DMA: instruction i of wave w fills stage rows 8 (w ND + i) .. + 7 (BMT = 1: waves 4-7 fill the rows of 0-3 again,
    // with the same bytes); lane l the 16 bytes at l, whose chunk the row's swizzle names
    const rsrc_t xr = make_rsrc(g.x + (int64_t)m0 * g.K, (uint32_t)((g.M - m0 < BM ? g.M - m0 : BM) * g.K * 2));
    uint32_t vo[ND], vl[ND];
    uint16_t* dst[ND];
#pragma unroll
    for (int i = 0; i < ND; ++i) {
        const int r0 = 8 * ((wave * ND + i) % (4 * BMT)), r = r0 + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
        vo[i] = m0 + r < g.M ? (uint32_t)(r * g.K + 8 * c) * 2u : OOB_VOFF;
        vl[i] = 64 * (IT - 1) + 8 * c < g.K ? vo[i] : OOB_VOFF;          // the last step's chunks past K read zero
        dst[i] = lds + r0 * RG_K;
    }
    // every step issues its weight loads and its DMA, past the end too (the last unit again; zeros into a stage that is not
    // read): the compiler then knows, on every path, which loads a wait covers
    auto dma = [&](int it, int stage) {
#pragma unroll
        for (int i = 0; i < ND; ++i)
            dma16(xr, dst[i] + stage * STAGE, it >= k1 ? OOB_VOFF : it == IT - 1 ? vl[i] : vo[i], (uint32_t)it * (RG_K * 2));
    };
    // a K of an odd number of units: the second half's unit past K is its last unit again (it meets zeros)
    auto unit = [&](int it) { const int u = 2 * (it < k1 ? it : k1 - 1) + half; return u < U ? u : U - 1; };

    f32x16_t acc[BMT];
#pragma unroll
    for (int r = 0; r < BMT; ++r)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[r][i] = 0.f;
    std::conditional_t<FACT, RawHalf<T>, RawRegs<T>> cur, nxt;
    auto load = [&](auto& d, int it) {
        if constexpr (FACT) raw_half_load<T>(d, row, it < k1 ? it : k1 - 1, half, U);
        else raw_load<T>(d, row, unit(it));
    };
    dma(k0, 0);
    asm volatile("" ::: "memory");
    load(cur, k0);
    asm volatile("" ::: "memory");
    dma(k0 + 1, 1);

    int st0 = 0, st2 = 2;                                                 // this step's stage; the one two steps on
    for (int it = k0; it < k1; ++it) {
        wait_vm<ND>();                                                    // all but the next stage's DMA has landed
        wait_lgkm0();                                                     // and the last step's reads of the stage DMA fills next
        barrier_nofence();
        load(nxt, it + 1);
        asm volatile("" ::: "memory");
        dma(it + 2, st2);
        const uint16_t* st = lds + st0 * STAGE;
        if constexpr (FACT) {
            constexpr int RT = BMT >= 2 ? 2 : 1, NG = 2 * BMT / RT;      // groups of RT row tiles, unit 0's then unit 1's
            const f32x16_t zero = {};
            bf16x8_t b[2];
            float s = 0.f, sp = 0.f;
            f32x16_t P[2][RT];
#pragma unroll
            for (int i = 0; i <= NG; ++i) {
                const int w = i / (NG / 2), r0 = i % (NG / 2) * RT;
                if (i < NG) {
                    sp = s;
                    if (r0 == 0) s = raw_half_codes<T>(cur, it, w, half, b);
#pragma unroll
                    for (int k = 0; k < 2; ++k)
#pragma unroll
                        for (int r = 0; r < RT; ++r) {
                            const bf16x8_t a = __builtin_bit_cast(bf16x8_t, ld16(st + rg_off(32 * (r0 + r) + col, 4 * w + 2 * k + half)));
                            P[i & 1][r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b[k], k == 0 ? zero : P[i & 1][r], 0, 0, 0);
                        }
                } else {
                    sp = s;
                }
                if (i > 0) {
                    const int q0 = (i - 1) % (NG / 2) * RT;
#pragma unroll
                    for (int r = 0; r < RT; ++r)
#pragma unroll
                        for (int e = 0; e < 16; ++e) acc[q0 + r][e] = __builtin_fmaf(sp, P[(i - 1) & 1][r][e], acc[q0 + r][e]);
                }
            }
        } else {
            const int u = unit(it);
            const RawScales sc = raw_scales<T>(cur, u);
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                float v[8];
                raw_vals<T>(cur, sc, u, s, v);
                bf16x8_t bt[NT], a[BMT];
                raw_split<NT>(v, bt);
#pragma unroll
                for (int r = 0; r < BMT; ++r) a[r] = __builtin_bit_cast(bf16x8_t, ld16(st + rg_off(32 * r + col, 4 * half + s)));
#pragma unroll
                for (int k = 0; k < NT; ++k)
#pragma unroll
                    for (int r = 0; r < BMT; ++r) acc[r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[r], bt[k], acc[r], 0, 0, 0);
            }
        }
        cur = nxt;
        st0 = st0 == 2 ? 0 : st0 + 1;
        st2 = st2 == 2 ? 0 : st2 + 1;
    }
    wait_vm<0>();                                                         // no DMA outlives the block's LDS

    if (p >= 0) {                                                         // a piece: its partial tile
        float* o = g.part + ((int64_t)p * BM + 4 * half) * RG_BN + wave * 32 + col;
#pragma unroll
        for (int r = 0; r < BMT; ++r)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[(32 * r + 8 * (i >> 2) + (i & 3)) * RG_BN] = acc[r][i];
        return;
    }
    uint32_t bad[(BMT + 1) / 2] = {};                                     // the lane's non-finite outputs, a bit each
    auto store = [&](auto bf16) {
#pragma unroll
        for (int r = 0; r < BMT; ++r)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int m = m0 + 32 * r + 8 * (i >> 2) + 4 * half + (i & 3);
                if (m < g.M && n < g.N) {
                    store_y(g.y, (int64_t)m * g.N + n, acc[r][i], decltype(bf16)::value);
                    bad[r >> 1] |= !(__builtin_fabsf(acc[r][i]) < __builtin_inff()) ? 1u << (16 * (r & 1) + i) : 0u;
                }
            }
    };
    if (g.out_bf16) store(std::true_type{});
    else store(std::false_type{});
    uint32_t any = 0;
#pragma unroll
    for (int i = 0; i < (BMT + 1) / 2; ++i) any |= bad[i];
    if (any == 0) return;
    for (int j = 0; j < 16 * BMT; ++j) {
        uint32_t w = 0;
#pragma unroll
        for (int i = 0; i < (BMT + 1) / 2; ++i) w = (j >> 5) == i ? bad[i] : w;
        if (!((w >> (j & 31)) & 1u)) continue;
        const int m = m0 + 32 * (j >> 4) + 8 * ((j >> 2) & 3) + 4 * half + (j & 3);
        store_y(g.y, (int64_t)m * g.N + n, raw_dot<T>(row, g.x + (int64_t)m * g.K, g.K), g.out_bf16);
    }
}

// the cut tiles' outputs: the S partials of each added in piece order (4 columns a thread), then y
template <int T>
__global__ __launch_bounds__(256) void raw_reduce_kernel(const RawGemmArgs g, int BM) {
    const int e = (int)(blockIdx.x * 256 + threadIdx.x) * 4, tile = g.full + blockIdx.y;
    const int m = (tile % g.tm) * BM + e / RG_BN, n0 = (tile / g.tm) * RG_BN + e % RG_BN;
    if (m >= g.M || n0 >= g.N) return;
    const float* q = g.part + (int64_t)blockIdx.y * g.S * BM * RG_BN + e;
    f32x4_t v = *reinterpret_cast<const f32x4_t*>(q);
    for (int s = 1; s < g.S; ++s) v += *reinterpret_cast<const f32x4_t*>(q + (int64_t)s * BM * RG_BN);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int n = n0 + i;
        if (n >= g.N) break;
        float f = v[i];
        if (!(__builtin_fabsf(f) < __builtin_inff())) f = raw_dot<T>(g.raw + (int64_t)n * raw_row_bytes<T>(g.K), g.x + (int64_t)m * g.K, g.K);
        store_y(g.y, (int64_t)m * g.N + n, f, g.out_bf16);
    }
}

// The plan of an (M, N, K) product: rows per tile, the tiles run whole and the cut of the rest.
struct RawPlan { int bmt, tm, tiles, full, S, ipp; };
static RawPlan raw_plan(int64_t M, int64_t N, int64_t K, int cus) {
    RawPlan p{};
    p.bmt = M <= 32 ? 1 : M <= 64 ? 2 : M <= 128 ? 4 : 8;
    p.tm = (int)((M + 32 * p.bmt - 1) / (32 * p.bmt));
    const int64_t tiles = p.tm * ((N + RG_BN - 1) / RG_BN), IT = (K + RG_K - 1) / RG_K;
    const int64_t P = (int64_t)cus;
    int64_t rem = tiles % P, best = 0, bs = 1;
    p.full = (int)(tiles - rem);
    // the rest in S pieces: the fewest K steps of the busiest CU, a piece's partial counted as two steps
    for (int64_t S = 1; rem > 0 && S <= 32 && S <= IT; ++S) {
        const int64_t ipp = (IT + S - 1) / S, pieces = rem * ((IT + ipp - 1) / ipp);
        const int64_t cost = (pieces + P - 1) / P * (ipp + (S > 1 ? 2 : 0)) + (S > 1 ? 4 : 0);
        if (S == 1 || cost < best) best = cost, bs = S;
    }
    if (rem == 0 || bs == 1) {
        p.full = (int)tiles;
        p.S = 1;
        p.ipp = (int)IT;
    } else {
        p.ipp = (int)((IT + bs - 1) / bs);
        p.S = (int)((IT + p.ipp - 1) / p.ipp);
    }
    p.tiles = (int)tiles;
    return p;
}

int64_t raw_gemm_work(int64_t M, int64_t N, int64_t K) {
    const RawPlan p = raw_plan(M, N, K, cus_of_device());
    return (int64_t)(p.tiles - p.full) * p.S * 32 * p.bmt * RG_BN * 4;
}

template <int T, int BMT>
static int raw_gemm_b(const RawGemmArgs& g, const RawPlan& p, hipStream_t s) {
    constexpr size_t lds = (size_t)3 * 32 * BMT * RG_K * 2;
    auto kern = raw_gemm_kernel<T, BMT>;
    static std::atomic<uint64_t> set{0};
    if (set_lds_limit((const void*)kern, lds, set) != hipSuccess) return set_error(MBQ_LAUNCH_FAIL, "raw GEMM: %zu bytes of LDS refused", lds);
    const int rem = p.tiles - p.full;
    kern<<<dim3((unsigned)(p.full + rem * p.S)), RG_T, lds, s>>>(g);
    if (rem > 0) raw_reduce_kernel<T><<<dim3((unsigned)(32 * BMT * RG_BN / 1024), (unsigned)rem), 256, 0, s>>>(g, 32 * BMT);
    return check_launch("raw GEMM");
}

template <int T>
static int raw_gemm_t(const uint8_t* raw, const uint16_t* x, int64_t M, int64_t N, int64_t K, void* y, int out_bf16, float* work,
                      hipStream_t s) {
    const RawPlan p = raw_plan(M, N, K, cus_of_device());
    const RawGemmArgs g{raw, x, y, work, (int)M, (int)N, (int)K, out_bf16, p.tm, p.full, p.S, p.ipp};
    switch (p.bmt) {
        case 1: return raw_gemm_b<T, 1>(g, p, s);
        case 2: return raw_gemm_b<T, 2>(g, p, s);
        case 4: return raw_gemm_b<T, 4>(g, p, s);
        default: return raw_gemm_b<T, 8>(g, p, s);
    }
}

int launch_raw_gemm(int t, const uint8_t* raw, const uint16_t* x, int64_t M, int64_t N, int64_t K, void* y, int out_bf16,
                    float* work, hipStream_t s) {
    switch (t) {
#define RAW_CASE(T) case T: return raw_gemm_t<T>(raw, x, M, N, K, y, out_bf16, work, s);
        RAW_CASE(T_F32) RAW_CASE(T_F16) RAW_CASE(T_BF16) RAW_CASE(T_Q4_1) RAW_CASE(T_Q5_0) RAW_CASE(T_Q5_1) RAW_CASE(T_Q2_K)
        RAW_CASE(T_Q3_K) RAW_CASE(T_IQ4_NL) RAW_CASE(T_IQ4_XS) RAW_CASE(T_TQ1_0) RAW_CASE(T_TQ2_0) RAW_CASE(T_MXFP4) RAW_CASE(T_NVFP4)
#undef RAW_CASE
    }
    return set_error(MBQ_BAD_ARG, "raw GEMM: no kernel for ggml type %d (kernel types run on their planes)", t);
}

}  // namespace mbq
