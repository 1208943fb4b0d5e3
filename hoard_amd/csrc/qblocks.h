// Device-side ggml K-quant super-block codecs for gfx950 (wave64).
//
// Formats (ggml-common.h, copied verbatim into the reference's expert slots,
// src/run_moe_stream.cpp:177-183):
//   block_q4_K 144 B: d fp16 | dmin fp16 | 12 B packed 6-bit scales+mins | 128 B nibbles
//   block_q6_K 210 B: ql[128] | qh[64] | int8 scales[16] | d fp16
//   block_q5_K 176 B: d fp16 | dmin fp16 | 12 B scales+mins as Q4_K | qh[32] | qs[128]
//   block_q3_K 110 B: hmask[32] | qs[64] (2-bit) | 12 B packed 6-bit scales | d fp16
//   block_q8_K 292 B: d f32 | int8 qs[256] | int16 bsums[16]   (activation side)
// Dot products are exact integer sums per super-block (v_dot4_i32_i8) scaled
// in fp32 exactly as the CPU path does: per block (d_w*d_x)*isum, and for
// Q4_K / Q5_K also (dmin_w*d_x)*msum, accumulated over blocks in block order.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hoard {

constexpr int QK = 256;
constexpr int kTypeQ3K = 11;
constexpr int kTypeQ4K = 12;
constexpr int kTypeQ5K = 13;
constexpr int kTypeQ6K = 14;
constexpr int kQ3KBytes = 110;
constexpr int kQ4KBytes = 144;
constexpr int kQ5KBytes = 176;
constexpr int kQ6KBytes = 210;

// Bytes of one super-block of a supported type (0 for any other).
__host__ __device__ constexpr int kquant_block_bytes(int type) {
    return type == kTypeQ4K ? kQ4KBytes
                            : type == kTypeQ6K ? kQ6KBytes
                                               : type == kTypeQ5K ? kQ5KBytes : type == kTypeQ3K ? kQ3KBytes : 0;
}
template <int T>
struct QType;
template <>
struct QType<kTypeQ4K> {
    static constexpr int bytes = kQ4KBytes;
    static constexpr bool has_min = true;
};
template <>
struct QType<kTypeQ6K> {
    static constexpr int bytes = kQ6KBytes;
    static constexpr bool has_min = false;
};
template <>
struct QType<kTypeQ5K> {
    static constexpr int bytes = kQ5KBytes;
    static constexpr bool has_min = true;
};
template <>
struct QType<kTypeQ3K> {
    static constexpr int bytes = kQ3KBytes;
    static constexpr bool has_min = false;
};

__device__ __forceinline__ float half_bits_to_float(uint32_t bits16) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)bits16);
}

// ggml's nearest_int (round to nearest even through the fp32 adder).
__device__ __forceinline__ int nearest_int(float f) {
    const float v = f + 12582912.0f;
    return (__float_as_int(v) & 0x007fffff) - 0x00400000;
}

__device__ __forceinline__ int sdot4(uint32_t a, uint32_t b, int c) {
    return __builtin_amdgcn_sdot4((int)a, (int)b, c, false);
}

// Q4_K scale/min pair for sub-block s from the 12 packed bytes (three words).
__device__ __forceinline__ void q4k_scale_min(int s, uint32_t s0, uint32_t s1, uint32_t s2, int &sc,
                                              int &mn) {
    // bytes 0..3 = s0, 4..7 = s1, 8..11 = s2
    auto byte = [&](int i) -> int {
        const uint32_t w = i < 4 ? s0 : (i < 8 ? s1 : s2);
        return (int)((w >> (8 * (i & 3))) & 0xffu);
    };
    if (s < 4) {
        sc = byte(s) & 63;
        mn = byte(s + 4) & 63;
    } else {
        sc = (byte(s + 4) & 0x0f) | ((byte(s - 4) >> 6) << 4);
        mn = (byte(s + 4) >> 4) | ((byte(s) >> 6) << 4);
    }
}

// Signed Q3_K scale g (stored as scale + 32 in 6 bits) from the 12 scale bytes
// held in words s0 (bytes 0..3), s1 (4..7), s2 (8..11).
__device__ __forceinline__ int q3k_scale(int g, uint32_t s0, uint32_t s1, uint32_t s2) {
    const uint32_t lw = (g & 4) ? s1 : s0;                   // byte g % 8
    const int lo = (int)((lw >> (8 * (g & 3) + ((g & 8) ? 4 : 0))) & 0x0fu);
    const int hi = (int)((s2 >> (8 * (g & 3) + 2 * (g >> 2))) & 3u);
    return (lo | (hi << 4)) - 32;
}

}  // namespace hoard
