// gfx950 (CDNA4) kernels of the quantized linear: dequant, device repack and the matmul dispatch (decode GEMV:
// mbq_gemv.hip; weight-stream GEMM: mbq_wsgemm.hip; LDS-tile MFMA GEMM: mbq_gemm.hip).
//
// Semantics follow reference src/mashbox/ops/__init__.py:594-632 (qmatmul: x @ W.T, float32 accumulation) with the
// weights of reference src/mashbox/ops/reference.py:66-70 (Q4_0), :101-103 (Q8_0), :132-149 (Q4_K), :150-159 (Q5_K) and
// :164-173 (Q6_K), and the int8 per-channel linear of reference src/mashbox/models/qwen3_8_27b/model.py:72-82. Plane layouts: mbq_layout.h.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>

#include "mbq_device.h"
#include "mbq_launch.h"
#include "mbq_layout.h"
#include "mbq_raw_unit.h"

namespace mbq {


// ------------------------------------------------------------------------------------------------------- dequant
// One thread per 16-byte unit (K-quants and Q4_0: 32 values; Q8_0: half a block, 16 values). Bit for bit the reference
// dequantization: Q8_0 v = f32(q) * d, Q4_0 v = d * f32(q - 8), Q4_K and Q5_K v = (d*sc)*q - dmin*m and
// Q6_K v = (d*sc)*(q - 32), whose products are exact in float32 (Q4_0 and Q6_K keep the reference's order of the
// operands, which fixes the sign of a zero).
// With `rows` (out_rows device row ids) it writes row r of w from weight row rows[r] (plus N when negative, clamped to
// [0, N - 1], as jax.numpy indexes): the rows of a lookup, without the rest of the weight. ids: ROWS_I32 as just said;
// ROWS_WRAP32 / ROWS_WRAP64 (int64 ids) plus N once more first (mbq_lookup_rows).
enum : int { ROWS_I32 = 0, ROWS_WRAP32 = 1, ROWS_WRAP64 = 2 };
template <int T>
__global__ __launch_bounds__(256) void dequant_kernel(const uint8_t* __restrict__ base, int64_t stride,
                                                      const int32_t* __restrict__ layer_dev, int nlayers, int64_t sc_off,
                                                      int64_t hi_off, int64_t d_off, int N, int K, float* __restrict__ w,
                                                      const void* __restrict__ rows, int ids, int64_t out_rows) {
    const int64_t uw = unit32(T) ? 32 : 16;
    const int64_t units = out_rows * (K / uw);
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= units) return;
    const int64_t lo = layer_offset(stride, layer_dev, nlayers);
    const bool ok = lo >= 0;
    base += ok ? lo : 0;
    const int64_t o = g / (K / uw), u = g % (K / uw);
    int64_t n = o;
    if (rows != nullptr) {
        n = ids == ROWS_WRAP64 ? static_cast<const int64_t*>(rows)[o] : static_cast<const int32_t*>(rows)[o];
        if (ids != ROWS_I32) n = (int32_t)(n < 0 ? n + N : n);
        n = n < 0 ? n + N : n;
        n = n < 0 ? 0 : (n >= N ? N - 1 : n);
    }
    float* out = w + o * K + u * uw;
    if (!ok) {
        for (int i = 0; i < uw; ++i) out[i] = __builtin_nanf("");
        return;
    }
    if constexpr (q6k_like(T)) {
        // T_Q6KT: unit u of chunk u / 4 in each tiled plane
        constexpr bool TL = T == T_Q6KT;
        const u32x4 q = ld16(base + (TL ? q4kt_off(n, K) + (u >> 2) * 1024 + (u & 3) * 16 : n * (K >> 1) + u * 16));
        const u32x2 h = *reinterpret_cast<const u32x2*>(base + hi_off + (TL ? q6kt_h_off(n, K) + (u >> 2) * 512 + (u & 3) * 8 : n * (K >> 2) + u * 8));
        const uint16_t scp = *reinterpret_cast<const uint16_t*>(base + sc_off + (TL ? q6kt_s_off(n, K) + (u >> 2) * 128 + (u & 3) * 2 : n * (K >> 4) + u * 2));
        const float d = f16f(*reinterpret_cast<const uint16_t*>(base + d_off + (TL ? q6kt_d_off(n, K) + (u >> 3) * 32 : (n * (K >> 8) + (u >> 3)) * 2)));
        const float ds0 = d * (float)(int8_t)(scp & 0xFFu), ds1 = d * (float)(int8_t)(scp >> 8);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            uint32_t lo, hi;
            q6k_bytes(q[t], h[t >> 1], t, &lo, &hi);
            const float ds = t < 2 ? ds0 : ds1;
            float v[8];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = ds * (float)((int)((lo >> (8 * e)) & 0xFFu) - 32);
                v[4 + e] = ds * (float)((int)((hi >> (8 * e)) & 0xFFu) - 32);
            }
            st16(out + t * 8, u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])});
            st16(out + t * 8 + 4, u32x4{__float_as_uint(v[4]), __float_as_uint(v[5]), __float_as_uint(v[6]), __float_as_uint(v[7])});
        }
    } else if constexpr (q5k_like(T)) {
        constexpr bool TL = T == T_Q5KT;                         // unit u of chunk u / 4 in each tiled plane
        const u32x4 q = ld16(base + (TL ? q4kt_off(n, K) + (u >> 2) * 1024 + (u & 3) * 16 : n * (K >> 1) + u * 16));
        const uint32_t h = *reinterpret_cast<const uint32_t*>(base + hi_off + (TL ? q5kt_h_off(n, K) + (u >> 2) * 256 + (u & 3) * 4 : n * (K >> 3) + u * 4));
        const u32x4 mt = ld16(base + sc_off + (TL ? q4kt_meta_off(n, K) + (u >> 3) * 256 : (n * (K >> 8) + (u >> 3)) * 16));
        uint32_t sc, mn;
        q4k_scale_min(mt[1], mt[2], mt[3], (int)(u & 7), &sc, &mn);
        const float dsc = f16f(mt[0]) * (float)sc;
        const float dm = f16f(mt[0] >> 16) * (float)mn;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            uint32_t lo, hi;
            q5k_bytes(q[t], h, t, &lo, &hi);
            float v[8];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = dsc * (float)((lo >> (8 * e)) & 0xFFu) - dm;
                v[4 + e] = dsc * (float)((hi >> (8 * e)) & 0xFFu) - dm;
            }
            st16(out + t * 8, u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])});
            st16(out + t * 8 + 4, u32x4{__float_as_uint(v[4]), __float_as_uint(v[5]), __float_as_uint(v[6]), __float_as_uint(v[7])});
        }
    } else if constexpr (q40_like(T)) {
        constexpr bool TL = T == T_Q40T;                         // block u: unit u % 4 of chunk u / 4 in the tiles
        const u32x4 q = ld16(base + (TL ? q40t_off(n, K) + (u >> 2) * 1024 + (u & 3) * 16 : n * (K >> 1) + u * 16));
        const float d = f16f(*reinterpret_cast<const uint16_t*>(base + sc_off + (TL ? q40t_d_off(n, K) + (u >> 2) * 128 + (u & 3) * 2 : (n * (K >> 5) + u) * 2)));
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int bit = 16 * (e & 1) + 4 * (e >> 1);
                v[e] = d * (float)((int)((q[t] >> bit) & 15u) - 8);
            }
            st16(out + t * 8, u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])});
            st16(out + t * 8 + 4, u32x4{__float_as_uint(v[4]), __float_as_uint(v[5]), __float_as_uint(v[6]), __float_as_uint(v[7])});
        }
    } else if constexpr (q4k_like(T)) {
        const u32x4 q = T == T_Q4KT ? ld16(base + q4kt_off(n, K) + (u >> 2) * 1024 + (u & 3) * 16) : ld16(base + n * (K >> 1) + u * 16);
        const u32x4 mt = T == T_Q4KT ? ld16(base + sc_off + q4kt_meta_off(n, K) + (u >> 3) * 256)
                                     : ld16(base + sc_off + (n * (K >> 8) + (u >> 3)) * 16);
        uint32_t sc, mn;
        q4k_scale_min(mt[1], mt[2], mt[3], (int)(u & 7), &sc, &mn);
        const float dsc = f16f(mt[0]) * (float)sc;
        const float dm = f16f(mt[0] >> 16) * (float)mn;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int bit = 16 * (e & 1) + 4 * (e >> 1);
                v[e] = dsc * (float)((q[t] >> bit) & 15u) - dm;
            }
            st16(out + t * 8, u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])});
            st16(out + t * 8 + 4, u32x4{__float_as_uint(v[4]), __float_as_uint(v[5]), __float_as_uint(v[6]), __float_as_uint(v[7])});
        }
    } else {
        // Q8_0 (T_Q8T: unit u's two 8-byte groups at their tile offsets; the scale of block u / 2 in the tiled d plane)
        u32x4 q;
        if constexpr (T == T_Q8T) {
            const uint8_t* c = base + i8t_off(n, K, (u >> 2) * 64) + q8t_byte((int)(u & 3) * 16);
            const u32x2 lo = *reinterpret_cast<const u32x2*>(c), hi = *reinterpret_cast<const u32x2*>(c + 16);
            q = u32x4{lo[0], lo[1], hi[0], hi[1]};
        } else {
            q = ld16(base + n * K + u * 16);
        }
        const float d = f16f(*reinterpret_cast<const uint16_t*>(
            base + sc_off + (T == T_Q8T ? q8t_d_off(n, K) + (u >> 2) * 64 + ((u >> 1) & 1) * 2 : (n * (K >> 5) + (u >> 1)) * 2)));
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = (float)(int8_t)(q[t] >> (8 * e)) * d;
            st16(out + t * 4, u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])});
        }
    }
}

// ------------------------------------------------------------------------------------------------- raw dequant
static int check_launch(const char* what);
// The file's blocks (rows, row_bytes) -> float32 (rows, cols), without planes: reference src/mashbox/ops/reference.py
// :398-409 (dequant) with :66-70 (Q4_0), :101-103 (Q8_0), :132-149 (Q4_K), :150-159 (Q5_K) and :164-173 (Q6_K), the
// rebuild of the exact path. One thread per 32 values (a Q4_0 / Q8_0 block, a Q4_K / Q5_K sub-block, two Q6_K
// sub-blocks); the blocks are 18 / 34 / 144 / 176 / 210 bytes apart, so bytes are read one at a time.
template <int T>
__global__ __launch_bounds__(256) void dequant_raw_kernel(const uint8_t* __restrict__ raw, int64_t rows, int K,
                                                          float* __restrict__ w) {
    const int64_t units = rows * (K / 32);
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= units) return;
    const int64_t n = g / (K / 32), u = g % (K / 32);
    float* out = w + n * K + u * 32;
    if constexpr (T == T_Q8_0) {
        const uint8_t* b = raw + (n * (K / 32) + u) * 34;
        const float d = f16f((uint32_t)b[0] | ((uint32_t)b[1] << 8));
        for (int i = 0; i < 32; ++i) out[i] = (float)(int8_t)b[2 + i] * d;
    } else if constexpr (T == T_Q4_0) {
        // value i < 16: low nibble of qs[i]; value 16 + i: its high nibble (qs at byte 2)
        const uint8_t* b = raw + (n * (K / 32) + u) * 18;
        const float d = f16f((uint32_t)b[0] | ((uint32_t)b[1] << 8));
        for (int i = 0; i < 32; ++i) out[i] = d * (float)((int)((b[2 + (i & 15)] >> (4 * (i >> 4))) & 15u) - 8);
    } else if constexpr (T == T_Q5_K) {
        // value 32j + i of the super-block: nibble j % 2 of qs[32 (j / 2) + i] (qs at byte 48), bit j of qh[i] (byte 16)
        const uint8_t* b = raw + (n * (K / 256) + (u >> 3)) * 176;
        const int j = (int)(u & 7);
        const uint32_t s0 = b[4] | (b[5] << 8) | (b[6] << 16) | ((uint32_t)b[7] << 24);
        const uint32_t s1 = b[8] | (b[9] << 8) | (b[10] << 16) | ((uint32_t)b[11] << 24);
        const uint32_t s2 = b[12] | (b[13] << 8) | (b[14] << 16) | ((uint32_t)b[15] << 24);
        uint32_t sc, mn;
        q4k_scale_min(s0, s1, s2, j, &sc, &mn);
        const float dsc = f16f((uint32_t)b[0] | ((uint32_t)b[1] << 8)) * (float)sc;      // exact
        const float dm = f16f((uint32_t)b[2] | ((uint32_t)b[3] << 8)) * (float)mn;       // exact
        for (int i = 0; i < 32; ++i) {
            const uint32_t q = ((b[48 + 32 * (j >> 1) + i] >> (4 * (j & 1))) & 15u) | (((b[16 + i] >> j) & 1u) << 4);
            out[i] = dsc * (float)q - dm;
        }
    } else if constexpr (T == T_Q6_K) {
        // value 32j + i of the super-block (j = 4g + r): nibble r / 2 of ql[64g + 32 (r % 2) + i], bits 2r, 2r + 1 of
        // qh[32g + i], sub-block scale sc[2j + i / 16]
        const uint8_t* b = raw + (n * (K / 256) + (u >> 3)) * 210;
        const int j = (int)(u & 7), g = j >> 2, r = j & 3;
        const float d = f16f((uint32_t)b[208] | ((uint32_t)b[209] << 8));
        const float ds0 = d * (float)(int8_t)b[192 + 2 * j], ds1 = d * (float)(int8_t)b[193 + 2 * j];
        for (int i = 0; i < 32; ++i) {
            const int q = ((b[64 * g + 32 * (r & 1) + i] >> (4 * (r >> 1))) & 15) | (((b[128 + 32 * g + i] >> (2 * r)) & 3) << 4);
            out[i] = (i < 16 ? ds0 : ds1) * (float)(q - 32);
        }
    } else {
        const uint8_t* b = raw + (n * (K / 256) + (u >> 3)) * 144;
        const int j = (int)(u & 7);
        const uint32_t s0 = b[4] | (b[5] << 8) | (b[6] << 16) | ((uint32_t)b[7] << 24);
        const uint32_t s1 = b[8] | (b[9] << 8) | (b[10] << 16) | ((uint32_t)b[11] << 24);
        const uint32_t s2 = b[12] | (b[13] << 8) | (b[14] << 16) | ((uint32_t)b[15] << 24);
        uint32_t sc, mn;
        q4k_scale_min(s0, s1, s2, j, &sc, &mn);
        const float dsc = f16f((uint32_t)b[0] | ((uint32_t)b[1] << 8)) * (float)sc;      // exact
        const float dm = f16f((uint32_t)b[2] | ((uint32_t)b[3] << 8)) * (float)mn;       // exact
        const uint8_t* q = b + 16 + 32 * (j >> 1);                   // sub-block 2g: low nibbles, 2g+1: high nibbles
        const int sh = (j & 1) * 4;
        for (int i = 0; i < 32; ++i) out[i] = dsc * (float)((q[i] >> sh) & 15u) - dm;
    }
}

// One thread per 32 values, as dequant_raw_kernel
template <int T>
__global__ __launch_bounds__(256) void dequant_raw_more_kernel(const uint8_t* __restrict__ raw, int64_t rows, int K,
                                                               float* __restrict__ w) {
    const int64_t units = rows * (K / 32);
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= units) return;
    const int64_t n = g / (K / 32), u = g % (K / 32);
    float v[32];
    raw_unit<T>(raw + n * raw_row_bytes<T>(K), (int)u, v);
    float* out = w + n * K + u * 32;
#pragma unroll
    for (int i = 0; i < 32; i += 4)
        st16(out + i, u32x4{__float_as_uint(v[i]), __float_as_uint(v[i + 1]), __float_as_uint(v[i + 2]), __float_as_uint(v[i + 3])});
}

// F32, F16, BF16 (reference :372-381): one value per block, any row length; the rows are contiguous in the file and
// in w, so one thread takes 4 consecutive values of the whole (rows x K) array
template <int T>
__global__ __launch_bounds__(256) void dequant_raw_float_kernel(const uint8_t* __restrict__ raw, int64_t total,
                                                                float* __restrict__ w) {
    const int64_t i0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    const int64_t i1 = i0 + 4 < total ? i0 + 4 : total;
    for (int64_t i = i0; i < i1; ++i) {
        if constexpr (T == T_F32) w[i] = __uint_as_float(le32(raw + 4 * i));
        else if constexpr (T == T_F16) w[i] = f16f(le16(raw + 2 * i));
        else w[i] = __uint_as_float(le16(raw + 2 * i) << 16);
    }
}

int launch_dequant_raw(int t, const uint8_t* raw, int64_t rows, int64_t K, float* w, hipStream_t s) {
    if (t == T_F32 || t == T_F16 || t == T_BF16) {
        const int64_t total = rows * K;
        const dim3 grid((unsigned)((total + 1023) / 1024));
        if (t == T_F32) dequant_raw_float_kernel<T_F32><<<grid, 256, 0, s>>>(raw, total, w);
        else if (t == T_F16) dequant_raw_float_kernel<T_F16><<<grid, 256, 0, s>>>(raw, total, w);
        else dequant_raw_float_kernel<T_BF16><<<grid, 256, 0, s>>>(raw, total, w);
        return check_launch("dequant_raw");
    }
    const int64_t units = rows * (K / 32);
    const dim3 grid((unsigned)((units + 255) / 256));
    switch (t) {
        case T_Q4_0: dequant_raw_kernel<T_Q4_0><<<grid, 256, 0, s>>>(raw, rows, (int)K, w); break;
        case T_Q4_K: dequant_raw_kernel<T_Q4_K><<<grid, 256, 0, s>>>(raw, rows, (int)K, w); break;
        case T_Q5_K: dequant_raw_kernel<T_Q5_K><<<grid, 256, 0, s>>>(raw, rows, (int)K, w); break;
        case T_Q6_K: dequant_raw_kernel<T_Q6_K><<<grid, 256, 0, s>>>(raw, rows, (int)K, w); break;
        case T_Q8_0: dequant_raw_kernel<T_Q8_0><<<grid, 256, 0, s>>>(raw, rows, (int)K, w); break;
        case T_Q4_1: dequant_raw_more_kernel<T_Q4_1><<<grid, 256, 0, s>>>(raw, rows, (int)K, w); break;
        case T_Q5_0: dequant_raw_more_kernel<T_Q5_0><<<grid, 256, 0, s>>>(raw, rows, (int)K, w); break;
        case T_Q5_1: dequant_raw_more_kernel<T_Q5_1><<<grid, 256, 0, s>>>(raw, rows, (int)K, w); break;
        case T_Q2_K: dequant_raw_more_kernel<T_Q2_K><<<grid, 256, 0, s>>>(raw, rows, (int)K, w); break;
        case T_Q3_K: dequant_raw_more_kernel<T_Q3_K><<<grid, 256, 0, s>>>(raw, rows, (int)K, w); break;
        case T_IQ4_NL: dequant_raw_more_kernel<T_IQ4_NL><<<grid, 256, 0, s>>>(raw, rows, (int)K, w); break;
        case T_IQ4_XS: dequant_raw_more_kernel<T_IQ4_XS><<<grid, 256, 0, s>>>(raw, rows, (int)K, w); break;
        case T_TQ1_0: dequant_raw_more_kernel<T_TQ1_0><<<grid, 256, 0, s>>>(raw, rows, (int)K, w); break;
        case T_TQ2_0: dequant_raw_more_kernel<T_TQ2_0><<<grid, 256, 0, s>>>(raw, rows, (int)K, w); break;
        case T_MXFP4: dequant_raw_more_kernel<T_MXFP4><<<grid, 256, 0, s>>>(raw, rows, (int)K, w); break;
        case T_NVFP4: dequant_raw_more_kernel<T_NVFP4><<<grid, 256, 0, s>>>(raw, rows, (int)K, w); break;
        default: return set_error(MBQ_BAD_ARG, "dequant_raw: no kernel for ggml type %d", t);
    }
    return check_launch("dequant_raw");
}

// -------------------------------------------------------------------------------------------------- zero fill
// n bytes at p set to zero, one byte per thread (the planes' alignment padding: under 256 bytes a run). A kernel, not
// hipMemsetAsync, so that a repack recorded into a HIP graph replays correctly.
__global__ __launch_bounds__(256) void zero_kernel(uint8_t* __restrict__ p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

int launch_zero(uint8_t* p, int64_t n, hipStream_t s) {
    if (n <= 0) return 0;
    zero_kernel<<<dim3((unsigned)((n + 255) / 256)), 256, 0, s>>>(p, n);
    return check_launch("zero fill");
}

// ------------------------------------------------------------------------------------------------ device repack
// One thread per block: the file's bytes (unaligned, 18, 34, 144, 176 or 210 bytes apart) into the planes of
// mbq_layout.h.
template <int T>
__global__ __launch_bounds__(256) void repack_kernel(const uint8_t* __restrict__ raw, int N, int K, uint8_t* __restrict__ planes,
                                                     int64_t sc_off, int64_t hi_off, int64_t d_off) {
    const int bv = (q8_like(T) || q40_like(T)) ? 32 : 256;
    const int bb = q40_like(T) ? 18 : q8_like(T) ? 34 : q4k_like(T) ? 144 : q5k_like(T) ? 176 : 210;
    const int64_t nb = K / bv;
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    // tiles: the last tile's padding rows too, and for T_Q8T / T_Q40T the padding blocks of the last chunk (written zero)
    const int64_t rows = tiled_type(T) ? ((int64_t)N + 15) / 16 * 16 : N;
    const int64_t nbr = T == T_Q8T ? ((int64_t)K + 63) / 64 * 2 : T == T_Q40T ? ((int64_t)K + 127) / 128 * 4 : nb;
    if (g >= rows * nbr) return;
    const int64_t n = g / nbr, b = g % nbr;
    const bool live = n < N && b < nb;
    const uint8_t* src = raw + (live ? n * nb * bb + b * bb : 0);
    if constexpr (T == T_Q8T) {
        uint8_t* q = planes + i8t_off(n, K, (32 * b) & ~int64_t(63));
        for (int i = 0; i < 32; ++i) q[q8t_byte(32 * (int)(b & 1) + i)] = live ? src[2 + i] : 0;
        uint8_t* d = planes + sc_off + q8t_d_off(n, K) + (b / 2) * 64 + (b % 2) * 2;
        d[0] = live ? src[0] : 0;
        d[1] = live ? src[1] : 0;
    } else if constexpr (T == T_Q8_0) {
        uint8_t* q = planes + n * K + b * 32;
        for (int i = 0; i < 32; ++i) q[i] = src[2 + i];
        uint8_t* d = planes + sc_off + (n * nb + b) * 2;
        d[0] = src[0];
        d[1] = src[1];
    } else if constexpr (q40_like(T)) {
        // T_Q40T: at the tile offsets; rows past N and blocks past K (the last chunk's padding) written zero
        constexpr bool TL = T == T_Q40T;
        uint8_t* d = planes + sc_off + (TL ? q40t_d_off(n, K) + (b >> 2) * 128 + (b & 3) * 2 : (n * nb + b) * 2);
        d[0] = live ? src[0] : 0;
        d[1] = live ? src[1] : 0;
        uint32_t* dst = reinterpret_cast<uint32_t*>(planes + (TL ? q40t_off(n, K) + (b >> 2) * 1024 + (b & 3) * 16 : n * (K >> 1) + b * 16));
        for (int t = 0; t < 4; ++t) {
            uint32_t v = 0;
            for (int e = 0; e < 8 && live; ++e) {
                const int i = t * 8 + e;                               // slot of mbq_layout.h: dword i/8, bits 16 (e&1) + 4 (e/2)
                v |= ((uint32_t)(src[2 + (i & 15)] >> (4 * (i >> 4))) & 15u) << (16 * (e & 1) + 4 * (e >> 1));
            }
            dst[t] = v;
        }
    } else if constexpr (q5k_like(T)) {
        // T_Q5KT: at the tile offsets; the last tile's rows past N written zero
        constexpr bool TL = T == T_Q5KT;
        uint8_t* meta = planes + sc_off + (TL ? q4kt_meta_off(n, K) + b * 256 : (n * nb + b) * 16);
        for (int i = 0; i < 16; ++i) meta[i] = live ? src[i] : 0;
        for (int j = 0; j < 8; ++j) {
            uint32_t* qd = reinterpret_cast<uint32_t*>(planes + (TL ? q4kt_off(n, K) + (2 * b + (j >> 2)) * 1024 + (j & 3) * 16 : n * (K >> 1) + b * 128 + j * 16));
            uint32_t* hd = reinterpret_cast<uint32_t*>(planes + hi_off + (TL ? q5kt_h_off(n, K) + (2 * b + (j >> 2)) * 256 + (j & 3) * 4 : n * (K >> 3) + b * 32 + j * 4));
            uint32_t qw[4] = {0, 0, 0, 0}, hw = 0;
            for (int i = 0; i < 32 && live; ++i) {
                const uint32_t lo = (src[48 + 32 * (j >> 1) + i] >> (4 * (j & 1))) & 15u;
                const uint32_t hi = (src[16 + i] >> j) & 1u;
                // slots of mbq_layout.h: low nibble dword i/8, byte i%4, bits 4 ((i/4)%2); high bit byte i%4,
                // bit 2 (i/8) + (i/4)%2
                qw[i >> 3] |= lo << (8 * (i & 3) + 4 * ((i >> 2) & 1));
                hw |= hi << (8 * (i & 3) + 2 * (i >> 3) + ((i >> 2) & 1));
            }
            for (int t = 0; t < 4; ++t) qd[t] = qw[t];
            hd[0] = hw;
        }
    } else if constexpr (q6k_like(T)) {
        // T_Q6KT: every plane's bytes at their tile offsets; the last tile's rows past N written zero
        constexpr bool TL = T == T_Q6KT;
        for (int i = 0; i < 16; ++i)
            planes[sc_off + (TL ? q6kt_s_off(n, K) + (2 * b + (i >> 3)) * 128 + (i & 7) : n * (K >> 4) + b * 16 + i)] = live ? src[192 + i] : 0;
        uint8_t* d = planes + d_off + (TL ? q6kt_d_off(n, K) + b * 32 : (n * nb + b) * 2);
        d[0] = live ? src[208] : 0;
        d[1] = live ? src[209] : 0;
        for (int j = 0; j < 8; ++j) {
            uint32_t* qd = reinterpret_cast<uint32_t*>(planes + (TL ? q4kt_off(n, K) + (2 * b + (j >> 2)) * 1024 + (j & 3) * 16 : n * (K >> 1) + b * 128 + j * 16));
            uint32_t* hd = reinterpret_cast<uint32_t*>(planes + hi_off + (TL ? q6kt_h_off(n, K) + (2 * b + (j >> 2)) * 512 + (j & 3) * 8 : n * (K >> 2) + b * 64 + j * 8));
            const int g = j >> 2, r = j & 3;
            uint32_t qw[4] = {0, 0, 0, 0}, hw[2] = {0, 0};
            for (int i = 0; i < 32 && live; ++i) {
                const uint32_t lo = (src[64 * g + 32 * (r & 1) + i] >> (4 * (r >> 1))) & 15u;
                const uint32_t hi = (src[128 + 32 * g + i] >> (2 * r)) & 3u;
                // slots of mbq_layout.h: low nibble dword i/8, byte i%4, bits 4 ((i/4)%2); high bits dword i/16,
                // byte i%4, bits 2 ((i/4)%4)
                qw[i >> 3] |= lo << (8 * (i & 3) + 4 * ((i >> 2) & 1));
                hw[i >> 4] |= hi << (8 * (i & 3) + 2 * ((i >> 2) & 3));
            }
            for (int t = 0; t < 4; ++t) qd[t] = qw[t];
            hd[0] = hw[0];
            hd[1] = hw[1];
        }
    } else if constexpr (T == T_Q4KT) {
        // the Q4_K units and header of row n at their tile offsets (mbq_layout.h); the rows of the last tile past the
        // weight's own (n >= N) are written zero
        uint8_t* meta = planes + sc_off + q4kt_meta_off(n, K) + b * 256;
        for (int i = 0; i < 16; ++i) meta[i] = live ? src[i] : 0;
        const uint8_t* qs = src + 16;
        for (int j = 0; j < 8; ++j) {
            uint32_t* dst = reinterpret_cast<uint32_t*>(planes + q4kt_off(n, K) + (2 * b + (j >> 2)) * 1024 + (j & 3) * 16);
            for (int t = 0; t < 4; ++t) {
                uint32_t v = 0;
                for (int e = 0; e < 8 && live; ++e) {
                    const int i = t * 8 + e;
                    const uint32_t byte = qs[32 * (j >> 1) + i];
                    const uint32_t q = (j & 1) ? (byte >> 4) : (byte & 15u);
                    v |= q << (16 * (e & 1) + 4 * (e >> 1));
                }
                dst[t] = v;
            }
        }
    } else {
        uint8_t* meta = planes + sc_off + (n * nb + b) * 16;
        for (int i = 0; i < 16; ++i) meta[i] = src[i];
        const uint8_t* qs = src + 16;
        uint32_t* dst = reinterpret_cast<uint32_t*>(planes + n * (K >> 1) + b * 128);
        for (int j = 0; j < 8; ++j)
            for (int t = 0; t < 4; ++t) {
                uint32_t v = 0;
                for (int e = 0; e < 8; ++e) {
                    const int i = t * 8 + e;
                    const uint32_t byte = qs[32 * (j >> 1) + i];
                    const uint32_t q = (j & 1) ? (byte >> 4) : (byte & 15u);
                    v |= q << (16 * (e & 1) + 4 * (e >> 1));
                }
                dst[j * 4 + t] = v;
            }
    }
}

// ------------------------------------------------------------------------------------------- tiled int8 repack
// One thread per 16 bytes of the quant plane (mbq_layout.h, T_I8T): thread g fills bytes 16 (g % 4) .. of row g / 4 % 16
// of block g / 64, from the row-major quants, or zero past N or K; the first NP threads also write the scale plane.
// HBM-bound, load-time only.
__global__ __launch_bounds__(256) void i8t_repack_kernel(const int8_t* __restrict__ q, const float* __restrict__ sc, int64_t N,
                                                         int64_t K, uint8_t* __restrict__ planes, int64_t sc_off, int64_t chunks,
                                                         int64_t np) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t kc_n = (K + 63) / 64;
    if (g < chunks) {
        const int64_t blk = g >> 6, c = g & 63, r = c >> 2, part = c & 3;
        const int64_t row = (blk / kc_n) * 16 + r, col = (blk % kc_n) * 64 + 16 * part;
        u32x4 v = {0u, 0u, 0u, 0u};
        if (row < N && col < K) v = ld16(q + row * K + col);           // K % 16 == 0: whole 16-byte pieces
        st16(planes + blk * 1024 + r * 64 + 16 * part, v);
    }
    if (g < np) reinterpret_cast<float*>(planes + sc_off)[g] = g < N ? sc[g] : 0.f;
}

int launch_i8t_repack(const int8_t* q, const float* sc, int64_t N, int64_t K, uint8_t* planes, const Layout& L, hipStream_t s) {
    const int64_t chunks = L.qs_bytes / 16, np = (N + 15) / 16 * 16;
    const int64_t threads = std::max(chunks, np);
    i8t_repack_kernel<<<dim3((unsigned)((threads + 255) / 256)), 256, 0, s>>>(q, sc, N, K, planes, L.sc_off, chunks, np);
    return check_launch("int8 repack");
}

// ------------------------------------------------------------------------------------------ int8 embedding rows
// y[t, :] = f32(q[r, :]) * s[r] (then rounded to bfloat16 when out_bf16), r = toks[t] (+ N when negative, clamped to
// [0, N - 1]): reference src/mashbox/models/qwen3_8_27b/model.py:132-139 (embed, whose int8_rows at :117-129 equals the
// plain gather bit for bit). HBM-bound: D bytes read and 2 D (4 D) written per token. VEC: D % 16 == 0, one thread per
// 16 values (one 16-byte load, two or four 16-byte stores); else one thread per value.
template <bool VEC>
__global__ __launch_bounds__(256) void embed_kernel(const int8_t* __restrict__ q, const float* __restrict__ s, int64_t N,
                                                    int64_t D, const int32_t* __restrict__ toks, void* __restrict__ y,
                                                    int out_bf16) {
    const int64_t t = blockIdx.y;
    int64_t r = toks[t];
    r = r < 0 ? r + N : r;
    r = r < 0 ? 0 : (r >= N ? N - 1 : r);
    const float sc = s[r];
    const int64_t per = VEC ? 16 : 1;
    const int64_t c = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * per;
    if (c >= D) return;
    if constexpr (VEC) {
        const u32x4 w = ld16(q + r * D + c);
        float v[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = (float)(int8_t)(w[e >> 2] >> (8 * (e & 3))) * sc;
        if (out_bf16) {
            uint16_t* o = reinterpret_cast<uint16_t*>(y) + t * D + c;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                u32x4 p;
#pragma unroll
                for (int e = 0; e < 4; ++e) p[e] = bf16_bits(v[8 * h + 2 * e]) | (bf16_bits(v[8 * h + 2 * e + 1]) << 16);
                st16(o + 8 * h, p);
            }
        } else {
            float* o = reinterpret_cast<float*>(y) + t * D + c;
#pragma unroll
            for (int h = 0; h < 4; ++h)
                st16(o + 4 * h, u32x4{__float_as_uint(v[4 * h]), __float_as_uint(v[4 * h + 1]), __float_as_uint(v[4 * h + 2]),
                                      __float_as_uint(v[4 * h + 3])});
        }
    } else {
        store_y(y, t * D + c, (float)q[r * D + c] * sc, out_bf16);
    }
}

int launch_int8_embed(const int8_t* q, const float* s, int64_t N, int64_t D, const int32_t* toks, int64_t T, void* y,
                      int out_bf16, hipStream_t st) {
    const bool vec = D % 16 == 0 && (reinterpret_cast<uintptr_t>(q) & 15) == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;
    const int64_t per = vec ? 16 : 1, threads = (D + per - 1) / per;
    const dim3 grid((unsigned)((threads + 255) / 256), (unsigned)T);
    if (vec)
        embed_kernel<true><<<grid, 256, 0, st>>>(q, s, N, D, toks, y, out_bf16);
    else
        embed_kernel<false><<<grid, 256, 0, st>>>(q, s, N, D, toks, y, out_bf16);
    return check_launch("int8 embed");
}

// -------------------------------------------------------------------------------------------------- launchers
static int check_launch(const char* what) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(MBQ_LAUNCH_FAIL, "%s: %s", what, hipGetErrorString(e));
    return 0;
}

// Decode batches (M <= GEMV_MAX_M) run the GEMV when it has a plan for the shape; a row too long for the activation
// rows' registers (e.g. K = 17408 at 3-4 rows, or a Q8_0 / int8 K over 24576) runs the weight-stream kernel instead,
// which takes any K (launch_gemm routes M <= GEMV_MAX_M there).
template <int T>
static int launch_t(const Args& a, hipStream_t s) {
    return a.M <= GEMV_MAX_M && gemv_runs(T, a) ? launch_gemv(T, a, s) : launch_gemm(T, a, s);
}

int cus_of_device() {
    static std::atomic<int> cache[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    int n = cache[dev].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cache[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

int launch_matmul(int t, const Args& a, hipStream_t s) {
    switch (t) {
        case T_Q4_0: return launch_t<T_Q4_0>(a, s);
        case T_Q8_0: return launch_t<T_Q8_0>(a, s);
        case T_Q4_K: return launch_t<T_Q4_K>(a, s);
        case T_Q5_K: return launch_t<T_Q5_K>(a, s);
        case T_Q6_K: return launch_t<T_Q6_K>(a, s);
        case T_INT8: return launch_t<T_INT8>(a, s);
        case T_I8T: return launch_t<T_I8T>(a, s);
        case T_Q4KT: return launch_t<T_Q4KT>(a, s);
        case T_Q8T: return launch_t<T_Q8T>(a, s);
        case T_Q6KT: return launch_t<T_Q6KT>(a, s);
        case T_Q5KT: return launch_t<T_Q5KT>(a, s);
        case T_Q40T: return launch_t<T_Q40T>(a, s);
    }
    return set_error(MBQ_BAD_ARG, "no kernel for type %d", t);
}

int launch_dequant(int t, const Args& a, float* w, const void* rows, int ids, int64_t out_rows, hipStream_t s) {
    const int64_t uw = unit32(t) ? 32 : 16;
    const int64_t units = (rows ? out_rows : a.N) * (a.K / uw);
    if (units == 0) return 0;
    const dim3 grid((unsigned)((units + 255) / 256));
    auto run = [&](auto kern) {
        kern<<<grid, 256, 0, s>>>(a.base, a.stride, a.layer_dev, a.nlayers, a.sc_off, a.hi_off, a.d_off, (int)a.N, (int)a.K, w,
                                  rows, ids, rows ? out_rows : a.N);
    };
    if (t == T_Q4_0) run(dequant_kernel<T_Q4_0>);
    else if (t == T_Q4_K) run(dequant_kernel<T_Q4_K>);
    else if (t == T_Q4KT) run(dequant_kernel<T_Q4KT>);
    else if (t == T_Q8T) run(dequant_kernel<T_Q8T>);
    else if (t == T_Q6KT) run(dequant_kernel<T_Q6KT>);
    else if (t == T_Q5KT) run(dequant_kernel<T_Q5KT>);
    else if (t == T_Q40T) run(dequant_kernel<T_Q40T>);
    else if (t == T_Q5_K) run(dequant_kernel<T_Q5_K>);
    else if (t == T_Q6_K) run(dequant_kernel<T_Q6_K>);
    else run(dequant_kernel<T_Q8_0>);
    return check_launch("dequant");
}

int launch_repack(int t, const uint8_t* raw, int64_t N, int64_t K, uint8_t* planes, const Layout& L, hipStream_t s) {
    const int64_t blocks = t == T_Q8T ? (N + 15) / 16 * 16 * ((K + 63) / 64 * 2)
                           : t == T_Q40T ? (N + 15) / 16 * 16 * ((K + 127) / 128 * 4)
                                      : (tiled_type(t) ? (N + 15) / 16 * 16 : N) * (K / block_values(t));
    const dim3 grid((unsigned)((blocks + 255) / 256));
    auto run = [&](auto kern) { kern<<<grid, 256, 0, s>>>(raw, (int)N, (int)K, planes, L.sc_off, L.hi_off, L.d_off); };
    if (t == T_Q4_0) run(repack_kernel<T_Q4_0>);
    else if (t == T_Q4_K) run(repack_kernel<T_Q4_K>);
    else if (t == T_Q4KT) run(repack_kernel<T_Q4KT>);
    else if (t == T_Q8T) run(repack_kernel<T_Q8T>);
    else if (t == T_Q6KT) run(repack_kernel<T_Q6KT>);
    else if (t == T_Q5KT) run(repack_kernel<T_Q5KT>);
    else if (t == T_Q40T) run(repack_kernel<T_Q40T>);
    else if (t == T_Q5_K) run(repack_kernel<T_Q5_K>);
    else if (t == T_Q6_K) run(repack_kernel<T_Q6_K>);
    else run(repack_kernel<T_Q8_0>);
    return check_launch("repack");
}

}  // namespace mbq
