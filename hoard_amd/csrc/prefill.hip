// Expert products of a batch: the counterpart of ggml_mul_mat_id over all T
// prompt tokens (src/run_m1.cpp:93-108) and of the verify step's mul_mat_id with
// per-token ids (src/run_specloop.cpp:126-139).
//
// batched.hip routes the tokens (or takes the caller's ids), forms Q8_K(fx)
// and sorts the (token, slot) pairs by (expert, token) into work units of one
// expert: of 4 pairs for the per-token dots of dotunits.h, of 16, 32 or 64 for
// the MFMA bodies here; the size of the expert's group decides, and one launch
// holds units of both of its batch's kinds.  Per MFMA unit:
//   gate/up  32 rows of gate and of up per workgroup (16 rows of one matrix per
//            wave) against the unit's tokens on v_mfma_i32_16x16x64_i8, 16
//            token columns per MFMA, the sub-block scales folded into the
//            weight operand; each weight super-block is loaded and folded once
//            and used for every token chunk of the unit; SwiGLU fused;
//   Q8_K(h)  per pair (by the down launch where that runs dots);
//   down     64 rows per workgroup; y goes to its (token, slot) place.
// Each (row, token) value is formed from the per-token path's integer sub-block
// sums in its fp32 order, so every token's result is the single-token path's bit
// for bit.
#include "dotunits.h"
#include "kernels.h"
#include "lds_dma.h"
#include "mfma.h"
#include "qblocks.h"
#include "rowdot.h"
#include "router_tail.h"

namespace hoard {

namespace {

constexpr int kWaveRows = 16;  // rows per wave: one MFMA tile
constexpr int kGuRows = 32;    // gate (and up) rows per workgroup: two 16-row tiles
constexpr int kDnRows = 64;    // down rows per workgroup

typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

__device__ __forceinline__ v4i mfma_16x16x64(v4i a, v4i b, v4i c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
}

// One Q4_K super-block of a 16-row tile, folded for v_mfma_i32_16x16x64_i8.
// Lane l supplies A[l % 16][16 g .. 16 g + 15] (g = l / 16) of each of the four
// MFMA steps (the lane layout checked by a probe: B[16 g ..][l % 16] alike,
// D[4 g + i][l % 16]).  Quant byte i of chunk q (32 bytes) holds element
// 64 q + i in its low nibble and 64 q + 32 + i in its high one (sub-blocks 2 q
// and 2 q + 1), and a step's K index is only a summation index: lane group g
// takes the whole of chunk g, as two 16-byte pieces p that each give two
// steps, step j = 2 p + h taking nibble half h of piece p, i.e. elements
// 64 g + 16 p + 32 h .. + 15 of sub-block 2 g + h.  Each quant byte is so
// loaded once (two 16-byte loads a lane), and the lane's B operand of step j
// is those 16 contiguous activation quants.  The sub-block scale sc (6 bits)
// is folded into A in two parts that keep every product an int8:
// hi = q * (sc >> 3) and lo = q * (sc & 7), each <= 105, with
// sc * q = 8 hi + lo; a nibble times a factor below 8 never carries into the
// next byte, so a whole word multiplies at once.  The min term
// sum_s m_s S_s (S_s the sum of sub-block s's activation quants) is one
// v_mfma_f32_16x16x32_f16 (min_operand below).  The chains give exactly the
// per-token path's integer sums isum = 8 D_hi + D_lo and msum = D_min.  Each
// 16-bit half of a word of four nibbles multiplies at once (v_pk_mul_lo_u16,
// full rate, where a 32-bit multiply is quarter rate).
struct Q4Fold {
    v4i hi[4], lo[4];
    v8h mn;
    float d[4], dmin[4];  // factors of the four rows whose results the lane receives
};

// The min term of a super-block as one fp16 MFMA.  Every part of a sub-block's
// sum S_s that the activation block stores (kSums32) and every
// min (6 bits) is an exact fp16, and the fp32 sum of 16 products stays below
// 8 * 63 * 4064 < 2^24, so msum comes out exact: K index 8 g + s holds the even
// parts (g = 0) and the low bits (g = 1) of the sums against m_s, and m = 0 at
// g = 2, 3, whose lanes read the sums again.  It replaces four int8 steps with
// m_s broadcast (12 -> 9 MFMAs per chunk step, and a conversion less per row).
// mn[0] / mn[1]: the mins of sub-blocks 0..3 / 4..7, a byte each.
__device__ __forceinline__ v8h min_operand(const uint32_t mn[2]) {
    const bool low = (threadIdx.x & 63) < 32;  // g = 0, 1
    typedef _Float16 v2h __attribute__((ext_vector_type(2)));
    const v2h k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
    v2h r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        // 0x6400 | m is 1024 + m; bytes 2 (i % 2) and 2 (i % 2) + 1 of the word, each below 0x64
        const uint32_t w = low ? mn[i >> 1] : 0u;
        r[i] = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, w, (i & 1) ? 0x04030402u : 0x04010400u)) - k1024;
    }
    return v8h{r[0][0], r[0][1], r[1][0], r[1][1], r[2][0], r[2][1], r[3][0], r[3][1]};
}
__device__ __forceinline__ v4f mfma_f16(v8h a, v8h b) {
    const v4f z = {0.0f, 0.0f, 0.0f, 0.0f};
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, z, 0, 0, 0);
}

typedef short v2s16 __attribute__((ext_vector_type(2)));
typedef unsigned short v2u16 __attribute__((ext_vector_type(2)));
// Bytes of w times f, byte by byte, where no product passes 255: none carries.
__device__ __forceinline__ int nib_mul(uint32_t w, uint32_t f) {
    const v2u16 m = {(unsigned short)f, (unsigned short)f};
    return (int)__builtin_bit_cast(uint32_t, __builtin_bit_cast(v2u16, w) * m);
}

// The lane's raw bytes of one super-block of a 16-row tile: its row's header
// and chunk g's 32 quant bytes; loaded one super-block ahead.  The fp16
// factors of the four rows whose results the lane receives come from those
// rows' lanes by a lane shuffle (four 4-byte gathers from global memory per
// super-block cost more than the shuffles).
struct Q4Raw {
    uint4 hd;
    uint4 qv[2];
};

__device__ __forceinline__ void q4_raw_load(const uint8_t *W, size_t rb, int b, Q4Raw &o) {
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const uint8_t *blk = W + (size_t)r * rb + (size_t)b * kQ4KBytes;
    o.hd = *reinterpret_cast<const uint4 *>(blk);
    o.qv[0] = *reinterpret_cast<const uint4 *>(blk + 16 + 32 * g);
    o.qv[1] = *reinterpret_cast<const uint4 *>(blk + 32 + 32 * g);
}

__device__ __forceinline__ void q4_fold(const Q4Raw &raw, Q4Fold &o) {
    const int g = (threadIdx.x & 63) >> 4;
    uint32_t sc[2], mn[2];
    q4k_scales_packed(raw.hd, sc, mn);
    // the scales and mins of sub-blocks 2 g (low nibbles) and 2 g + 1 (high)
    const int s0 = 2 * g;
    const uint32_t sc0 = (uint32_t)byte_of(sc[s0 >> 2], s0 & 3), sc1 = (uint32_t)byte_of(sc[s0 >> 2], (s0 & 3) + 1);
    o.mn = min_operand(mn);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint4 qv = raw.qv[j >> 1];
        const uint32_t nsh = 4u * (uint32_t)(j & 1), scs = (j & 1) ? sc1 : sc0;
        const uint32_t w[4] = {(qv.x >> nsh) & 0x0f0f0f0fu, (qv.y >> nsh) & 0x0f0f0f0fu, (qv.z >> nsh) & 0x0f0f0f0fu,
                               (qv.w >> nsh) & 0x0f0f0f0fu};
        const uint32_t h = scs >> 3, lw = scs & 7u;
        o.hi[j] = v4i{nib_mul(w[0], h), nib_mul(w[1], h), nib_mul(w[2], h), nib_mul(w[3], h)};
        o.lo[j] = v4i{nib_mul(w[0], lw), nib_mul(w[1], lw), nib_mul(w[2], lw), nib_mul(w[3], lw)};
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t dm = (uint32_t)__shfl((int)raw.hd.x, 4 * g + i);
        o.d[i] = half_bits_to_float(dm & 0xffffu);
        o.dmin[i] = half_bits_to_float(dm >> 16);
    }
}

// The lane's operands of one token's activation block: four 16-byte pieces of
// its quants (which ones depends on the fold), its sums (types with a min
// term) and its scale.
struct XOps {
    v4i x[4];
    v8h bs;
    float xd;
};

// acc / accm of the lane's four rows for one super-block: the integer sums
// from the MFMA chains, then the per-token path's fp32 block terms in order.
__device__ __forceinline__ void q4_fold_step(const Q4Fold &w, const XOps &x, float acc[4], float accm[4]) {
    v4i dh = {0, 0, 0, 0}, dl = {0, 0, 0, 0};
    const v4f dn = mfma_f16(w.mn, x.bs);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        dh = mfma_16x16x64(w.hi[j], x.x[j], dh);
        dl = mfma_16x16x64(w.lo[j], x.x[j], dl);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int isum = 8 * dh[i] + dl[i];
        const float dd = w.d[i] * x.xd;
        const float dm = w.dmin[i] * x.xd;
        acc[i] = acc[i] + dd * (float)isum;
        accm[i] = accm[i] + dm * dn[i];
    }
}
// Step j of a Q4_K fold takes activation quants 64 g + 16 (j / 2) + 32 (j % 2) .. + 15.
template <class X>
__device__ __forceinline__ void q4_load_x(const X &x, XOps &o) {
    const int g = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) o.x[j] = *reinterpret_cast<const v4i *>(&x.qs[16 * g + 4 * (j >> 1) + 8 * (j & 1)]);
}
template <class X>
__device__ __forceinline__ v8h load_sums(const X &x) {
    return reinterpret_cast<const v8h *>(x.bsums)[((threadIdx.x & 63) >> 4) & 1];
}

// The same operand from a block whose sums are int16 (kSumsInt): b, its sixteen
// 16-element sums; half: which v8h (load_sums).  Q3_K takes the sums as they are
// (kSums16), the others the 32-element sums in two parts (kSums32).
template <int TG>
__device__ __forceinline__ v8h sums_from_int(const v4i (&b)[2], int half) {
    v8h r;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        if constexpr (TG == kTypeQ3K) {
            const int w = half ? b[1][s >> 1] : b[0][s >> 1];
            r[s] = (_Float16)(float)((s & 1) ? w >> 16 : (int)(int16_t)w);
        } else {
            const int w = b[s >> 2][s & 3], v = (int)(int16_t)w + (w >> 16);
            r[s] = (_Float16)(float)(half ? v & 1 : v & ~1);
        }
    }
    return r;
}

// -- Q8_K of h per sorted pair --------------------------------------------------
// grid (pairs), block 64 * NBH: wave b quantises block b of the pair's h.
__global__ __launch_bounds__(256) void pf_quant_h_kernel(BatchedArgs a) {
    const int pos = blockIdx.x, b = wave_index();
    const int nbh = a.n_ff / QK;
    if (b >= nbh) return;
    const float d = wave_quantize_q8l<kSums32>(a.hbuf + (size_t)pos * a.n_ff + (size_t)b * QK,
                                      reinterpret_cast<Q8L *>(a.q8h) + (size_t)pos * nbh + b);
    // the scales again, four to a pair: the down kernels copy a unit's in one 16-byte load a lane
    if ((threadIdx.x & 63) == 0) a.q8hd[(size_t)pos * 4 + b] = d;
}

// Bytes 0, 2 and 1, 3 of w in the 16-bit halves of two words, and back.
__device__ __forceinline__ void bytes_to_halves(uint32_t w, uint32_t &w02, uint32_t &w13) {
    w02 = __builtin_amdgcn_perm(0u, w, 0x0c020c00u);
    w13 = __builtin_amdgcn_perm(0u, w, 0x0c030c01u);
}
__device__ __forceinline__ int halves_to_bytes(uint32_t w02, uint32_t w13) {
    return (int)__builtin_amdgcn_perm(w13, w02, 0x06020400u);
}
// The high bytes of the halves.
__device__ __forceinline__ int high_bytes(uint32_t w02, uint32_t w13) {
    return (int)__builtin_amdgcn_perm(w13, w02, 0x07030501u);
}

// -- down, Q6_K rows folded for v_mfma_i32_16x16x64_i8 --------------------------
// Lane l of a wave supplies A[l % 16][16 g .. + 15] (g = l / 16) of each 64-element
// chunk jc of a super-block: elements 64 jc + 16 g .. + 15 of row l % 16, whose
// 6-bit values are nibble (jc % 2) of ql bytes 64 (jc / 2) + 16 g .. + 15 with
// bits 4 (jc % 2) + 2 (g / 2) .. + 1 of qh bytes 128 + 32 (jc / 2) + 16 (g % 2) ..
// + 15 on top, and which share one group scale, sc = scales[4 jc + g].  The
// per-token path forms isum = sum_g sc_g * sum_{e in g} (q_e - 32) x_e.  Here
// w = sc * (q - 32) = sc * q - 32 sc (one 16-bit multiply-add; -4064 <= w <=
// 4096) is split as w = 256 hi + lo with lo its low byte read as int8 and
// hi = (w + 128) >> 8 in [-16, 16]: isum = 256 D_hi + D_lo, exactly, and both
// parts are bytes of 16-bit words as they stand.  A super-block of the tile is
// folded once and used for every token chunk of the unit.  (With the zero
// point as a third MFMA chain, sc broadcast, a step took 12 MFMAs for these 8.)
struct Q6Fold {
    v4i hi[4], lo[4];
    float d[4];  // factors of the four rows whose results the lane receives
};

// 16 bytes at a 2-byte aligned address in memory, which takes such loads at any
// width, and in LDS.
__device__ __forceinline__ uint4 mem_u128_a2(const uint8_t *p) {
    typedef uint32_t v4u_a2 __attribute__((ext_vector_type(4), aligned(2)));
    const v4u_a2 v = *reinterpret_cast<const v4u_a2 *>(p);
    return make_uint4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ uint4 lds_u128_a2(const uint8_t *p) {
    const uint2 a = lds_u64_a2(p), b = lds_u64_a2(p + 8);
    return make_uint4(a.x, a.y, b.x, b.y);
}

// The lane's raw bytes of the block: its ql and qh pieces of both halves, the
// scales of its groups, its row's factor; from LDS or from memory.
struct Q6Raw {
    uint4 ql[2], qh[2];
    int sc[4];
    uint32_t d;
};
__device__ __forceinline__ void raw_lds(const uint8_t *T, size_t rb, int b, Q6Raw &o) {
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const uint8_t *blk = T + (size_t)r * rb + (size_t)b * kQ6KBytes;
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        o.ql[n] = lds_u128_a2(blk + 64 * n + 16 * g);
        o.qh[n] = lds_u128_a2(blk + 128 + 32 * n + 16 * (g & 1));
    }
#pragma unroll
    for (int jc = 0; jc < 4; ++jc) o.sc[jc] = (int)(int8_t)blk[192 + 4 * jc + g];
    o.d = (uint32_t)*reinterpret_cast<const uint16_t *>(blk + 208);
}
__device__ __forceinline__ void raw_load(const uint8_t *W, size_t rb, int b, Q6Raw &o) {
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const uint8_t *blk = W + (size_t)r * rb + (size_t)b * kQ6KBytes;
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        o.ql[n] = mem_u128_a2(blk + 64 * n + 16 * g);
        o.qh[n] = mem_u128_a2(blk + 128 + 32 * n + 16 * (g & 1));
    }
    const uint4 sc = mem_u128_a2(blk + 192);
    const uint32_t scw[4] = {sc.x, sc.y, sc.z, sc.w};
#pragma unroll
    for (int jc = 0; jc < 4; ++jc) o.sc[jc] = (int)(int8_t)(scw[jc] >> (8 * g));
    o.d = *reinterpret_cast<const uint16_t *>(blk + 208);
}

__device__ __forceinline__ void fold(const Q6Raw &raw, Q6Fold &o) {
    const int g = (threadIdx.x & 63) >> 4;
    const uint32_t h2 = 2u * (uint32_t)(g >> 1);
#pragma unroll
    for (int jc = 0; jc < 4; ++jc) {
        const uint4 ql = raw.ql[jc >> 1], qh = raw.qh[jc >> 1];
        const int sc = raw.sc[jc];
        const v2s16 s2 = {(short)sc, (short)sc}, z2 = {(short)(128 - 32 * sc), (short)(128 - 32 * sc)};
        const uint32_t qlw[4] = {ql.x, ql.y, ql.z, ql.w}, qhw[4] = {qh.x, qh.y, qh.z, qh.w};
        int hw[4], lw[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            // the upper two bits, at 2 (g / 2) or 4 + 2 (g / 2) of each byte, moved to bits 4 and 5
            const uint32_t up = ((jc & 1) ? qhw[k] >> h2 : qhw[k] << (4u - h2)) & 0x30303030u;
            const uint32_t q = ((qlw[k] >> (4 * (jc & 1))) & 0x0f0f0f0fu) | up;
            // w + 128 in 16-bit halves (bytes 0, 2 and 1, 3): the high byte is hi,
            // the low one lo with its top bit turned
            uint32_t q02, q13;
            bytes_to_halves(q, q02, q13);
            const uint32_t a02 = __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2s16, q02) * s2 + z2);
            const uint32_t a13 = __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2s16, q13) * s2 + z2);
            lw[k] = (int)((uint32_t)halves_to_bytes(a02, a13) ^ 0x80808080u);
            hw[k] = high_bytes(a02, a13);
        }
        o.hi[jc] = v4i{hw[0], hw[1], hw[2], hw[3]};
        o.lo[jc] = v4i{lw[0], lw[1], lw[2], lw[3]};
    }
    // the factors of the lane's four result rows, from the lanes that hold those rows
#pragma unroll
    for (int i = 0; i < 4; ++i) o.d[i] = half_bits_to_float((uint32_t)__shfl((int)raw.d, 4 * g + i));
}

// The quants of one token's block as the Q3_K, Q5_K and Q6_K folds take them:
// step jc elements 64 jc + 16 g .. + 15.
template <class X>
__device__ __forceinline__ void q6_load_x(const X &x, XOps &o) {
    const int g = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int jc = 0; jc < 4; ++jc) o.x[jc] = *reinterpret_cast<const v4i *>(&x.qs[16 * jc + 4 * g]);
}

__device__ __forceinline__ void fold_step(const Q6Fold &w, const XOps &x, float acc[4], float *) {
    v4i dh = {0, 0, 0, 0}, dl = {0, 0, 0, 0};
#pragma unroll
    for (int jc = 0; jc < 4; ++jc) {
        dh = mfma_16x16x64(w.hi[jc], x.x[jc], dh);
        dl = mfma_16x16x64(w.lo[jc], x.x[jc], dl);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int isum = 256 * dh[i] + dl[i];
        acc[i] = acc[i] + (w.d[i] * x.xd) * (float)isum;
    }
}

// Q3_K super-block b of a 16-row tile (110-byte blocks, only 2-byte aligned), folded for v_mfma_i32_16x16x64_i8.  Lane group
// g of chunk jc supplies elements 64 jc + 16 g .. + 15 of its row: 32-element
// range 2 jc + g / 2 (half n = jc / 2, quarter j = 2 (jc & 1) + g / 2),
// positions l = 16 (g & 1) .. + 15, one 16-element scale group G = 4 jc + g.
// Its quants are q3 = q - 4, q = q2 + 4 h (q2: bits 2 j .. 2 j + 1 of
// qs[32 n + l]; h: bit 4 n + j of hmask[l]), its scale sc_G is in [-32, 31].
// sc_G * q3 reaches 128, but w = sc_G * (q3 + 1) lies in [-128, 124], an int8, so
// one MFMA chain forms sum w x, and what the 1 adds comes off through an fp16
// MFMA over the 16-element sums T_G (exact: at most 2032):
// isum = D_w - sum_G sc_G T_G.  Five MFMAs a chunk step and 16 registers, where
// sc * q3 split in two int8 parts takes eight and 32.
struct Q3Fold {
    v4i w[4];
    v8h sc;      // -sc of the groups of the lane's K range (zero at g = 2, 3)
    float d[4];  // factors of the four rows whose results the lane receives
};
// The lane's raw bytes of the block: its half of hmask, its half of the qs of
// both 128-element halves, its row's scales and factor.
struct Q3Raw {
    uint4 hm, qv[2];
    uint32_t s[3], d;
};
__device__ __forceinline__ void raw_load(const uint8_t *W, size_t rb, int b, Q3Raw &o) {
    typedef uint32_t v3u_a2 __attribute__((ext_vector_type(3), aligned(2)));
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const uint8_t *blk = W + (size_t)r * rb + (size_t)b * kQ3KBytes;
    const v3u_a2 sc = *reinterpret_cast<const v3u_a2 *>(blk + 96);
    o.hm = mem_u128_a2(blk + 16 * (g & 1));
    o.qv[0] = mem_u128_a2(blk + 32 + 16 * (g & 1));
    o.qv[1] = mem_u128_a2(blk + 64 + 16 * (g & 1));
    o.s[0] = sc[0];
    o.s[1] = sc[1];
    o.s[2] = sc[2];
    o.d = *reinterpret_cast<const uint16_t *>(blk + 108);
}

__device__ __forceinline__ void fold(const Q3Raw &raw, Q3Fold &o) {
    const uint32_t g = (threadIdx.x & 63) >> 4, gh = g >> 1;
    // scale bytes g of the three words: groups g, 4 + g, 8 + g, 12 + g
    const uint32_t b0 = raw.s[0] >> (8 * g), b1 = raw.s[1] >> (8 * g), b2 = raw.s[2] >> (8 * g);
    const uint32_t s6[4] = {(b0 & 15u) | ((b2 & 3u) << 4), (b1 & 15u) | ((b2 & 12u) << 2),
                            ((b0 >> 4) & 15u) | (b2 & 48u), ((b1 >> 4) & 15u) | ((b2 >> 2) & 48u)};
    const uint32_t hm[4] = {raw.hm.x >> gh, raw.hm.y >> gh, raw.hm.z >> gh, raw.hm.w >> gh};
#pragma unroll
    for (int jc = 0; jc < 4; ++jc) {
        const int n = jc >> 1, cq = 4 * (jc & 1), ch = 4 * n + 2 * (jc & 1);  // after the lane's own shifts
        const uint4 &qv = raw.qv[n];
        const uint32_t qw[4] = {qv.x >> (2 * gh), qv.y >> (2 * gh), qv.z >> (2 * gh), qv.w >> (2 * gh)};
        const int sc = (int)s6[jc] - 32;
        const v2s16 scv = {(short)sc, (short)sc}, z = {(short)(-3 * sc), (short)(-3 * sc)};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t h = ch < 2 ? hm[k] << (2 - ch) : hm[k] >> (ch - 2);  // the bit at bit 2 of each byte
            const uint32_t q = ((qw[k] >> cq) & 0x03030303u) | (h & 0x04040404u);
            uint32_t q02, q13;
            bytes_to_halves(q, q02, q13);
            o.w[jc][k] = halves_to_bytes(__builtin_bit_cast(uint32_t, __builtin_bit_cast(v2s16, q02) * scv + z),
                                         __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2s16, q13) * scv + z));
        }
    }
    // the scales of groups 8 g .. 8 g + 7 (g = 0, 1) as fp16: 0x6400 | s is 1024 + s
    typedef _Float16 v2h __attribute__((ext_vector_type(2)));
    const uint32_t sh = 4u * (g & 1u);
    uint32_t w0 = ((raw.s[0] >> sh) & 0x0f0f0f0fu) | (((raw.s[2] >> sh) & 0x03030303u) << 4);
    uint32_t w1 = ((raw.s[1] >> sh) & 0x0f0f0f0fu) | (((raw.s[2] >> sh) & 0x0c0c0c0cu) << 2);
    w0 = g < 2 ? w0 : 0x20202020u;  // sc = 0
    w1 = g < 2 ? w1 : 0x20202020u;
    const v2h k1056 = {(_Float16)1056.0f, (_Float16)1056.0f};
    v2h r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t w = i < 2 ? w0 : w1;
        r[i] = k1056 - __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, w, (i & 1) ? 0x04030402u : 0x04010400u));
    }
    o.sc = v8h{r[0][0], r[0][1], r[1][0], r[1][1], r[2][0], r[2][1], r[3][0], r[3][1]};
#pragma unroll
    for (int i = 0; i < 4; ++i) o.d[i] = half_bits_to_float((uint32_t)__shfl((int)raw.d, 4 * (int)g + i));
}

__device__ __forceinline__ void fold_step(const Q3Fold &w, const XOps &x, float acc[4], float *) {
    v4i dw = {0, 0, 0, 0};
    const v4f dt = mfma_f16(w.sc, x.bs);
#pragma unroll
    for (int jc = 0; jc < 4; ++jc) dw = mfma_16x16x64(w.w[jc], x.x[jc], dw);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int isum = dw[i] + (int)dt[i];
        acc[i] = acc[i] + (w.d[i] * x.xd) * (float)isum;
    }
}

// Q5_K super-block b of a 16-row tile (16-byte aligned 176-byte blocks: d, dmin, Q4_K-packed scales and mins, qh[32], qs[128]), folded as the Q4_K
// gate/up tile is: lane group g of chunk jc takes nibble g / 2 of qs bytes
// 32 jc + 16 (g & 1) .. + 15 with bit 2 jc + g / 2 of qh[l] on top (q5 in
// [0, 31]), sub-block s = 2 jc + g / 2.  sc_s is taken two bits at a time, so
// that q5 * part (at most 93) stays a byte of a word multiply:
// isum = 16 D_2 + 4 D_1 + D_0; the min term is Q4_K's fp16 MFMA.  (Two chains
// of a product formed in 16-bit halves cost 5 vector instructions more per
// word of four quants.)
struct Q5Fold {
    v4i p[3][4];
    v8h mn;
    float d[4], dmin[4];  // factors of the four rows whose results the lane receives
};

// The lane's raw bytes of the block: its row's header, its half of qh (l = 16 (g & 1)
// .. + 15) and of each chunk's qs; from LDS or from memory.
struct Q5Raw {
    uint4 hd, qh, qv[4];
};
__device__ __forceinline__ void raw_load(const uint8_t *W, size_t rb, int b, Q5Raw &o) {
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const uint8_t *blk = W + (size_t)r * rb + (size_t)b * kQ5KBytes;
    o.hd = *reinterpret_cast<const uint4 *>(blk);
    o.qh = *reinterpret_cast<const uint4 *>(blk + 16 + 16 * (g & 1));
#pragma unroll
    for (int jc = 0; jc < 4; ++jc) o.qv[jc] = *reinterpret_cast<const uint4 *>(blk + 48 + 32 * jc + 16 * (g & 1));
}

__device__ __forceinline__ void fold(const Q5Raw &raw, Q5Fold &o) {
    const int g = (threadIdx.x & 63) >> 4;
    const uint4 hd = raw.hd, qh = raw.qh;
    uint32_t sc[2], mn[2];
    q4k_scales_packed(hd, sc, mn);
    const uint32_t qhw[4] = {qh.x, qh.y, qh.z, qh.w};
    const uint32_t nsh = 4u * (uint32_t)(g >> 1), bsh = 8u * (uint32_t)(g >> 1);
    o.mn = min_operand(mn);
    const uint32_t qh1[4] = {qhw[0] >> (g >> 1), qhw[1] >> (g >> 1), qhw[2] >> (g >> 1), qhw[3] >> (g >> 1)};
#pragma unroll
    for (int jc = 0; jc < 4; ++jc) {
        const uint32_t sh = 16u * (uint32_t)(jc & 1) + bsh;  // byte 2 (jc & 1) + g / 2 of word jc / 2
        const uint32_t scs = (sc[jc >> 1] >> sh) & 0xffu;
        const uint4 qv = raw.qv[jc];
        const uint32_t qw[4] = {qv.x, qv.y, qv.z, qv.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            // the fifth bit, bit s = 2 jc + g / 2 of each qh byte, moved to bit 4
            const uint32_t up = (jc < 2 ? qh1[k] << (4 - 2 * jc) : qh1[k] >> (2 * jc - 4)) & 0x10101010u;
            const uint32_t q = ((qw[k] >> nsh) & 0x0f0f0f0fu) | up;
            o.p[0][jc][k] = nib_mul(q, scs & 3u);
            o.p[1][jc][k] = nib_mul(q, (scs >> 2) & 3u);
            o.p[2][jc][k] = nib_mul(q, scs >> 4);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t dm = (uint32_t)__shfl((int)hd.x, 4 * g + i);  // from the lanes that hold those rows
        o.d[i] = half_bits_to_float(dm & 0xffffu);
        o.dmin[i] = half_bits_to_float(dm >> 16);
    }
}

__device__ __forceinline__ void fold_step(const Q5Fold &w, const XOps &x, float acc[4], float accm[4]) {
    v4i d0 = {0, 0, 0, 0}, d1 = {0, 0, 0, 0}, d2 = {0, 0, 0, 0};
    const v4f dn = mfma_f16(w.mn, x.bs);
#pragma unroll
    for (int jc = 0; jc < 4; ++jc) {
        d0 = mfma_16x16x64(w.p[0][jc], x.x[jc], d0);
        d1 = mfma_16x16x64(w.p[1][jc], x.x[jc], d1);
        d2 = mfma_16x16x64(w.p[2][jc], x.x[jc], d2);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int isum = 4 * (4 * d2[i] + d1[i]) + d0[i];
        const float dd = w.d[i] * x.xd;
        const float dm = w.dmin[i] * x.xd;
        acc[i] = acc[i] + dd * (float)isum;
        accm[i] = accm[i] + dm * dn[i];
    }
}

// A type's super-block of a 16-row tile: the lane's raw bytes from memory (load)
// or from LDS (lds), their fold, and the fold's operands.
template <int T>
struct Tile;
template <>
struct Tile<kTypeQ4K> {
    using Raw = Q4Raw;
    using Fold = Q4Fold;
    static __device__ __forceinline__ void load(const uint8_t *W, size_t rb, int b, Raw &o) { q4_raw_load(W, rb, b, o); }
    static __device__ __forceinline__ void lds(const uint8_t *t, size_t rb, int b, Raw &o) { q4_raw_load(t, rb, b, o); }
    static __device__ __forceinline__ void fold(const Raw &r, Fold &o) { q4_fold(r, o); }
    static __device__ __forceinline__ void load_x(const Q8L &x, XOps &o) {
        q4_load_x(x, o);
        o.bs = load_sums(x);
    }
    static __device__ __forceinline__ void step(const Fold &w, const XOps &x, float acc[4], float accm[4]) {
        q4_fold_step(w, x, acc, accm);
    }
};
template <>
struct Tile<kTypeQ5K> {
    using Raw = Q5Raw;
    using Fold = Q5Fold;
    static __device__ __forceinline__ void load(const uint8_t *W, size_t rb, int b, Raw &o) { raw_load(W, rb, b, o); }
    static __device__ __forceinline__ void lds(const uint8_t *t, size_t rb, int b, Raw &o) { raw_load(t, rb, b, o); }
    static __device__ __forceinline__ void fold(const Raw &r, Fold &o) { hoard::fold(r, o); }
    static __device__ __forceinline__ void load_x(const Q8L &x, XOps &o) {
        q6_load_x(x, o);
        o.bs = load_sums(x);
    }
    static __device__ __forceinline__ void step(const Fold &w, const XOps &x, float acc[4], float accm[4]) {
        fold_step(w, x, acc, accm);
    }
};
template <>
struct Tile<kTypeQ6K> {
    using Raw = Q6Raw;
    using Fold = Q6Fold;
    static __device__ __forceinline__ void load(const uint8_t *W, size_t rb, int b, Raw &o) { raw_load(W, rb, b, o); }
    static __device__ __forceinline__ void lds(const uint8_t *t, size_t rb, int b, Raw &o) { raw_lds(t, rb, b, o); }
    static __device__ __forceinline__ void fold(const Raw &r, Fold &o) { hoard::fold(r, o); }
    static __device__ __forceinline__ void load_x(const Q8L &x, XOps &o) { q6_load_x(x, o); }
    static __device__ __forceinline__ void step(const Fold &w, const XOps &x, float acc[4], float accm[4]) {
        fold_step(w, x, acc, accm);
    }
};

// The gate/up row types: a lane's raw bytes of a super-block of a 16-row tile
// from memory, its fold, the fold's operands and step.  pin(): the fold is done
// before the loads that follow (or their registers are copied every step).
template <int TG>
struct GateUp;
template <>
struct GateUp<kTypeQ4K> {
    using Raw = Q4Raw;
    using Fold = Q4Fold;
    static constexpr int kDepth = 3;
    static __device__ __forceinline__ void load(const uint8_t *W, size_t rb, int b, Raw &o) { q4_raw_load(W, rb, b, o); }
    static __device__ __forceinline__ void fold(const Raw &r, Fold &o) { q4_fold(r, o); }
    template <class X>
    static __device__ __forceinline__ void load_x(const X &x, XOps &o) {
        q4_load_x(x, o);
    }
    static __device__ __forceinline__ void step(const Fold &w, const XOps &x, float acc[4], float accm[4]) {
        q4_fold_step(w, x, acc, accm);
    }
    static __device__ __forceinline__ void pin(const Fold &f) {
        asm volatile("" ::"v"(f.hi[0]), "v"(f.hi[1]), "v"(f.hi[2]), "v"(f.hi[3]), "v"(f.lo[0]), "v"(f.lo[1]),
                     "v"(f.lo[2]), "v"(f.lo[3])
                     : "memory");
    }
};
template <>
struct GateUp<kTypeQ3K> {
    using Raw = Q3Raw;
    using Fold = Q3Fold;
    static constexpr int kDepth = 3;
    static __device__ __forceinline__ void load(const uint8_t *W, size_t rb, int b, Raw &o) { raw_load(W, rb, b, o); }
    static __device__ __forceinline__ void fold(const Raw &r, Fold &o) { hoard::fold(r, o); }
    template <class X>
    static __device__ __forceinline__ void load_x(const X &x, XOps &o) {
        q6_load_x(x, o);
    }
    static __device__ __forceinline__ void step(const Fold &w, const XOps &x, float acc[4], float accm[4]) {
        fold_step(w, x, acc, accm);
    }
    static __device__ __forceinline__ void pin(const Fold &f) {
        asm volatile("" ::"v"(f.w[0]), "v"(f.w[1]), "v"(f.w[2]), "v"(f.w[3]), "v"(f.sc) : "memory");
    }
};
// -- gate/up + SwiGLU ------------------------------------------------------------
// 32 rows of gate and of up per workgroup: wave w takes rows [32 x + 16 (w % 2), +16)
// of gate (w < 2) or up (w >= 2) of the unit's expert against every token of the
// unit.  Per super-block the workgroup copies the Q8_K blocks of the unit's
// token chunks into LDS (one buffer ahead) while each wave holds the next
// super-block of its rows in registers; the gate waves hand their values to the
// up waves through LDS, which form h and store it to hbuf[sorted pair][row].
// Bound by its vector and matrix instructions, which share a SIMD's issue (53 of
// 88 us a launch without any load, Qwen3-30B at 512 tokens, 226 MB), and by loads
// that arrive later than one super-block ahead covers (the other 35).  Q3_K rows
// took 174 us at 512 tokens of 64 experts with a tile in LDS and every wave
// loading its tokens' blocks, 115 here.
// LDS: xs, two buffers of the unit's Q8_K block b; gx, the gate values [row
// tile][chunk][row i][lane].  CH: the 16-token chunks of a unit.  kInt: the blocks'
// sums are int16 (a batch that runs dots too).
constexpr int kXGran = (int)sizeof(Q8L) / 16;  // 16-byte granules staged per token
template <int CH>
constexpr int kLargeXBytes = 2 * 16 * CH * (int)sizeof(Q8L);
template <int CH>
constexpr int kLargeGxBytes = 2 * CH * 4 * 64 * (int)sizeof(float);

template <int TG, int NB, int CH, bool kInt>
__device__ __forceinline__ void gateup_large(const BatchedArgs &a, const Unit &w, uint8_t *smem) {
    using S = GateUp<TG>;
    constexpr int kTok = 16 * CH;
    constexpr int kXChunksPerBlock = (kTok * kXGran + 63) / 64;  // 1 KB copies per unit block
    Q8L(*xs)[kTok] = reinterpret_cast<Q8L(*)[kTok]>(smem);
    float(*gx)[CH][4][64] = reinterpret_cast<float(*)[CH][4][64]>(smem + kLargeXBytes<CH>);
    const int wave = wave_index(), lane = threadIdx.x & 63, c = lane & 15, q = lane >> 4;
    const int m = wave >> 1, rt = wave & 1;
    const int row0 = blockIdx.x * kGuRows + rt * kWaveRows;
    constexpr size_t rb = (size_t)NB * QType<TG>::bytes;
    const uint8_t *W = (m ? batched_up(a, w.e) : batched_gate(a, w.e)) + (size_t)row0 * rb;
    const int nch = (w.n + 15) >> 4;
    // this lane's granules of the x copy: chunks wave, wave + 4, ...; only the
    // unit's tokens are copied (the MFMA columns of the places past them read
    // whatever the buffer holds, and their results are not stored)
    constexpr int kXJ = (kXChunksPerBlock + 3) / 4;
    const int ngran = w.n * kXGran;
    // byte offsets into q8x (it holds at most 512 tokens' blocks): half the
    // registers of pointers
    uint32_t xoff[kXJ];
#pragma unroll
    for (int j = 0; j < kXJ; ++j) {
        const int p = 64 * (wave + 4 * j) + lane, tt = min(p / kXGran, kTok - 1), o = p % kXGran;
        xoff[j] = (uint32_t)a.ptok[w.p0 + min(tt, w.n - 1)] * (uint32_t)(NB * sizeof(Q8L)) + 16u * o;
    }
    auto stage_x = [&](int b, int buf) {
#pragma unroll
        for (int j = 0; j < kXJ; ++j) {
            const int ck = wave + 4 * j;
            if (64 * ck < ngran && 64 * ck + lane < ngran)
                dma_lanes(reinterpret_cast<uint8_t *>(&xs[buf][0]) + 1024 * ck,
                          a.q8x + (xoff[j] + (uint32_t)(b * sizeof(Q8L))));
        }
    };
    float acc[CH][4], accm[CH][4];
#pragma unroll
    for (int ch = 0; ch < CH; ++ch)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[ch][i] = accm[ch][i] = 0.0f;
    typename S::Raw raw;
    S::load(W, rb, 0, raw);
    stage_x(0, 0);
#pragma unroll 1
    for (int b = 0; b < NB; ++b) {
        // Other waves read the x chunks this wave copied: the compiler does not
        // see the copies, so the wave waits for its own before the barrier (it
        // waits for the raw weight loads of block b there anyway).
        lds_dma_wait();
        __syncthreads();  // every wave's copies of x(b) landed, and x(b - 1) is read
        typename S::Fold t;
        S::fold(raw, t);
        S::pin(t);
        // the next super-block's activation copies issue before its weight
        // loads (both are waited for at the next super-block; copies first
        // measured 3 % faster for the layer at 512 tokens)
        if (b + 1 < NB) {
            stage_x(b + 1, (b + 1) & 1);
            S::load(W, rb, b + 1, raw);
        }
        const Q8L *xb = xs[b & 1];
#pragma unroll
        for (int ch = 0; ch < CH; ++ch)
            if (ch < nch) {
                const Q8L &x = xb[ch * 16 + c];
                XOps xo;
                S::load_x(x, xo);
                if constexpr (kInt) {
                    const v4i *b2 = reinterpret_cast<const v4i *>(x.bsums), s2[2] = {b2[0], b2[1]};
                    xo.bs = sums_from_int<TG>(s2, q & 1);
                } else {
                    xo.bs = load_sums(x);
                }
                xo.xd = x.d;
                S::step(t, xo, acc[ch], accm[ch]);
            }
    }
    if (m == 0) {
#pragma unroll
        for (int ch = 0; ch < CH; ++ch)
#pragma unroll
            for (int i = 0; i < 4; ++i) gx[rt][ch][i][lane] = acc[ch][i] - accm[ch][i];
    }
    __syncthreads();
    if (m == 0) return;
#pragma unroll
    for (int ch = 0; ch < CH; ++ch) {
        const int idx = ch * 16 + c;
        if (ch < nch && idx < w.n) {
            float hv[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float g = gx[rt][ch][i][lane], uu = acc[ch][i] - accm[ch][i];
                hv[i] = g / (1.0f + expf(-g)) * uu;
            }
            *reinterpret_cast<float4 *>(a.hbuf + (size_t)(w.p0 + idx) * a.n_ff + row0 + 4 * q) =
                make_float4(hv[0], hv[1], hv[2], hv[3]);
        }
    }
}

// -- gate/up + SwiGLU for units of at most 16 pairs ------------------------------
// Rows and waves as above.  With one token chunk a wave's registers leave room
// for kDepth super-blocks of raw weights in flight, and all of the unit's
// activation blocks fit LDS at once (39 KB, four workgroups a CU): one barrier
// after they land, then every wave streams its rows from memory at its own
// pace.  Qwen3.5 at 131 tokens (302 MB): 85 -> 72 us a launch against units of
// 64; Q3_K at 27 tokens 75 (per-token dots) -> 54.
// The quants and scale of a Q8_K block in LDS (17 granules: 16 tokens' reads
// of one place fall into different banks).
struct Q8S {
    int32_t qs[64];
    float d;
    int32_t pad[3];
};
static_assert(sizeof(Q8S) == 272 && offsetof(Q8L, d) == 288 && offsetof(Q8L, bsums) == 256, "Q8S from Q8L");
template <int NB>
constexpr int kSmallLds = NB * 16 * (int)sizeof(Q8S) + NB * 32 * 16;

template <int TG, int NB, bool kInt>
__device__ __forceinline__ void gateup_small(const BatchedArgs &a, const Unit &w, uint8_t *smem) {
    using S = GateUp<TG>;
    constexpr int D = S::kDepth, kGran = (int)sizeof(Q8S) / 16, kCopies = (16 * kGran + 63) / 64;
    static_assert(NB % 4 == 0 && NB >= D, "a wave copies NB / 4 blocks of every token");
    Q8S(*xs)[16] = reinterpret_cast<Q8S(*)[16]>(smem);
    v4i(*sums)[32] = reinterpret_cast<v4i(*)[32]>(smem + NB * 16 * sizeof(Q8S));
    const int wave = wave_index(), lane = threadIdx.x & 63, c = lane & 15, q = lane >> 4;
    const int m = wave >> 1, rt = wave & 1;
    const int row0 = blockIdx.x * kGuRows + rt * kWaveRows;
    constexpr size_t rb = (size_t)NB * QType<TG>::bytes;
    const uint8_t *W = (m ? batched_up(a, w.e) : batched_gate(a, w.e)) + (size_t)row0 * rb;
    // the tokens of this lane's granules, then the first weights, then the copies
    int tk[kCopies + 1];
#pragma unroll
    for (int j = 0; j <= kCopies; ++j) {
        const int tt = j < kCopies ? (64 * j + lane) / kGran : lane >> 1;
        tk[j] = a.ptok[w.p0 + min(tt, w.n - 1)];
    }
    asm volatile("" ::: "memory");
    typename S::Raw raw[D];
#pragma unroll
    for (int i = 0; i < D; ++i) S::load(W, rb, i, raw[i]);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < NB / 4; ++i) {
        const int b = wave * (NB / 4) + i;
        const uint32_t blk = (uint32_t)(b * (int)sizeof(Q8L));
#pragma unroll
        for (int j = 0; j < kCopies; ++j) {
            const int p = 64 * j + lane, o = p % kGran;
            if (64 * j < w.n * kGran && p < w.n * kGran)
                dma_lanes(reinterpret_cast<uint8_t *>(&xs[b][0]) + 1024 * j,
                          a.q8x + ((uint32_t)tk[j] * (uint32_t)(NB * sizeof(Q8L)) + blk + 16u * (o < 16 ? o : 18)));
        }
        if (lane < 2 * w.n)
            dma_lanes(reinterpret_cast<uint8_t *>(&sums[b][0]),
                      a.q8x + ((uint32_t)tk[kCopies] * (uint32_t)(NB * sizeof(Q8L)) + blk + 256u + 16u * (lane & 1)));
    }
    lds_dma_wait();
    __syncthreads();
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f}, accm[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        typename S::Fold f;
        S::fold(raw[b % D], f);
        S::pin(f);  // the fold is done before its registers are loaded again
        if (b + D < NB) S::load(W, rb, b + D, raw[b % D]);
        const Q8S &x = xs[b][c];
        XOps xo;
        xo.xd = x.d;
        if constexpr (kInt) {
            const v4i s2[2] = {sums[b][2 * c], sums[b][2 * c + 1]};
            xo.bs = sums_from_int<TG>(s2, q & 1);
        } else {
            xo.bs = __builtin_bit_cast(v8h, sums[b][2 * c + (q & 1)]);
        }
        S::load_x(x, xo);
        S::step(f, xo, acc, accm);
    }
    // the gate waves hand their values to the up waves over the activations
    __syncthreads();
    float *gx = reinterpret_cast<float *>(&xs[0][0]) + (size_t)rt * 256;
    if (m == 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) gx[64 * i + lane] = acc[i] - accm[i];
    }
    __syncthreads();
    if (m == 0 || c >= w.n) return;
    float hv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float g = gx[64 * i + lane], uu = acc[i] - accm[i];
        hv[i] = g / (1.0f + expf(-g)) * uu;
    }
    *reinterpret_cast<float4 *>(a.hbuf + (size_t)(w.p0 + c) * a.n_ff + row0 + 4 * q) =
        make_float4(hv[0], hv[1], hv[2], hv[3]);
}

// grid (n_ff / 32, max units), block 256.  With kRows = 16 rows of a dot unit per
// workgroup it is (n_ff / 16, max units) and an MFMA unit leaves the upper half of
// the row blocks idle.
template <int TG, int NB, int kRows>
__global__ __launch_bounds__(256, 4) void gateup_dots_kernel(BatchedArgs a) {
    using Dots = DotGateUp<TG, NB>;
    __shared__ __align__(16) uint8_t smem[Dots::kLds > kSmallLds<NB> ? Dots::kLds : kSmallLds<NB>];
    Unit w;
    if (!load_unit(a, blockIdx.y, w)) return;
    if (w.dots) {
#pragma unroll 1
        for (int r = 0; r < kRows; r += kDotGuRows) {
            if (r > 0) __syncthreads();  // every wave is done with the rows before
            Dots::run(a, w, blockIdx.x * kRows + r, smem);
        }
    } else if (kRows != kGuRows) {
        if ((int)blockIdx.x * kGuRows < a.n_ff) gateup_small<TG, NB, true>(a, w, smem);
    } else if (w.n <= 16) {
        gateup_small<TG, NB, true>(a, w, smem);
    } else {
        gateup_large<TG, NB, 2, true>(a, w, smem);
    }
}
template <int TG, int NB>
__global__ __launch_bounds__(256, 4) void gateup_mixed_kernel(BatchedArgs a) {
    constexpr int CH = 2;
    static_assert(kSmallLds<NB> >= kLargeXBytes<CH> + kLargeGxBytes<CH>, "both units' LDS");
    __shared__ __align__(16) uint8_t smem[kSmallLds<NB>];
    Unit w;
    if (!load_unit(a, blockIdx.y, w)) return;
    if (w.n <= 16)
        gateup_small<TG, NB, false>(a, w, smem);
    else
        gateup_large<TG, NB, CH, false>(a, w, smem);
}
// Three workgroups share a CU (47 KB of LDS each).
template <int TG, int NB>
__global__ __launch_bounds__(256, 3) void gateup_large_kernel(BatchedArgs a) {
    __shared__ __align__(16) uint8_t smem[kLargeXBytes<4> + kLargeGxBytes<4>];
    Unit w;
    if (load_unit(a, blockIdx.y, w)) gateup_large<TG, NB, 4, false>(a, w, smem);
}

// -- down: 64 rows of the unit's expert, y to its (token, slot) place -----------
// block 256.  Each wave copies its own 16 rows into LDS in one burst and waits
// for them alone (no barrier before the folds); each super-block of them is
// folded once, then run against every token chunk of a pass (CH of 16 pairs).
// TS: the shared expert's row type beside routed rows of type TD (Qwen3.5: Q6_K
// beside Q5_K), in the same launch.
// With four chunks, Q6_K keeps two operand sets (chunk ch's loaded while the one
// before it computes, three workgroups a CU); Q4_K and Q5_K load every chunk's
// before the fold, which covers them, and one chunk always is.
template <int T, int NBH, int CH>
__device__ __forceinline__ void down_rows16(const uint8_t *tile, int nch, const Q8L *x0, const int (&xi)[CH],
                                            const float (*xds)[4], float (&acc)[CH][4], float (&accm)[CH][4]) {
    using K = Tile<T>;
    const int c = threadIdx.x & 15;
    auto load_x = [&](int ch, int b, XOps &o) {
        K::load_x(x0[(size_t)xi[ch] * NBH + b], o);
        o.xd = xds[ch * 16 + c][b];
    };
#pragma unroll 1
    for (int b = 0; b < NBH; ++b) {
        typename K::Raw raw;
        typename K::Fold f;
        if constexpr (T == kTypeQ6K && CH == 4) {
            XOps xa, xb;
            load_x(0, b, xa);
            K::lds(tile, NBH * QType<T>::bytes, b, raw);
            K::fold(raw, f);
            if (nch > 1) load_x(1, b, xb);
            K::step(f, xa, acc[0], accm[0]);
            if (nch > 1) {
                if (nch > 2) load_x(2, b, xa);
                K::step(f, xb, acc[1], accm[1]);
                if (nch > 2) {
                    if (nch > 3) load_x(3, b, xb);
                    K::step(f, xa, acc[2], accm[2]);
                    if (nch > 3) K::step(f, xb, acc[3], accm[3]);
                }
            }
        } else {
            XOps xc[CH];
#pragma unroll
            for (int ch = 0; ch < CH; ++ch)
                if (ch < nch) load_x(ch, b, xc[ch]);
            K::lds(tile, NBH * QType<T>::bytes, b, raw);
            K::fold(raw, f);
#pragma unroll
            for (int ch = 0; ch < CH; ++ch)
                if (ch < nch) K::step(f, xc[ch], acc[ch], accm[ch]);
        }
    }
}

// kPairs: the most pairs of a unit; CH, CHS: the chunks of a pass over the tile,
// of routed rows and of the shared expert's (a unit of more takes several
// passes, its rows folded again for each).
template <int TD, int NBH, int TS, int kPairs, int CH, int CHS = CH>
struct DownTile {
    static constexpr int kRowBytesD = NBH * QType<TD>::bytes, kRowBytesS = NBH * QType<TS>::bytes;
    static_assert(kWaveRows * kRowBytesD % 16 == 0 && kWaveRows * kRowBytesS % 16 == 0, "16-byte copies");
    // LDS: the tile, y row (token * slots + slot) of each of the unit's pairs,
    // each wave's copy of the pairs' Q8_K(h) scales
    static constexpr int kTileBytes = kDnRows * (kRowBytesD > kRowBytesS ? kRowBytesD : kRowBytesS);
    static constexpr int kLds = kTileBytes + kPairs * (int)sizeof(int) + 4 * kPairs * 4 * (int)sizeof(float);

    template <int T, int C>
    static __device__ __forceinline__ void passes(const BatchedArgs &a, const Unit &w, const uint8_t *tile,
                                                  const int *yrow, const float (*xds)[4], int row0) {
        const int lane = threadIdx.x & 63, c = lane & 15, q = lane >> 4;
        const Q8L *x0 = reinterpret_cast<const Q8L *>(a.q8h) + (size_t)w.p0 * NBH;
        constexpr bool kOne = kPairs == 16 * C;
        if (!kOne) __syncthreads();  // yrow is written
#pragma unroll 1
        for (int p0 = 0; p0 < w.n; p0 += 16 * C) {
            const int nch = min((w.n - p0 + 15) >> 4, C);
            int xi[C];  // the lane's pair of each chunk (places past the last repeat it)
#pragma unroll
            for (int ch = 0; ch < C; ++ch) xi[ch] = min(p0 + ch * 16 + c, w.n - 1);
            float acc[C][4], accm[C][4];
#pragma unroll
            for (int ch = 0; ch < C; ++ch)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[ch][i] = accm[ch][i] = 0.0f;
            down_rows16<T, NBH, C>(tile, nch, x0, xi, xds + p0, acc, accm);
            if (kOne) __syncthreads();  // yrow is written
#pragma unroll
            for (int ch = 0; ch < C; ++ch) {
                const int idx = p0 + ch * 16 + c;
                if (ch < nch && idx < w.n) {
                    // accm stays 0 for rows without a min term
                    *reinterpret_cast<float4 *>(a.ybuf + (size_t)yrow[idx] * a.n_embd + row0 + 4 * q) =
                        make_float4(acc[ch][0] - accm[ch][0], acc[ch][1] - accm[ch][1], acc[ch][2] - accm[ch][2],
                                    acc[ch][3] - accm[ch][3]);
                }
            }
            if (kOne) break;
        }
    }

    static __device__ __forceinline__ void run(const BatchedArgs &a, const Unit &w, uint8_t *smem) {
        int *yrow = reinterpret_cast<int *>(smem + kTileBytes);
        float(*xds)[kPairs][4] = reinterpret_cast<float(*)[kPairs][4]>(yrow + kPairs);
        const bool shx = TS != TD && a.sh && w.e == a.n_ids;  // the shared expert's rows
        const int wave = wave_index(), lane = threadIdx.x & 63, tid = threadIdx.x;
        const int row0 = blockIdx.x * kDnRows + wave * kWaveRows;
        // the pairs' places, read while the tile lands
        const int pt = tid < w.n ? a.ptok[w.p0 + tid] : 0, ps = tid < w.n ? a.pslot[w.p0 + tid] : 0;
        const int wbytes = kWaveRows * (shx ? kRowBytesS : kRowBytesD);
        uint8_t *T = smem + wave * wbytes;
        // the pairs' block scales with the tile: a 4-byte load of a scale with every
        // chunk's quants cost more
        if (kPairs == 64 || lane < kPairs)
            dma_lanes(reinterpret_cast<uint8_t *>(&xds[wave][0][0]),
                      reinterpret_cast<const uint8_t *>(a.q8hd + (size_t)(w.p0 + min(lane, w.n - 1)) * 4));
        dma_wave_copy_nt(T, batched_down(a, w.e) + (size_t)row0 * (wbytes / kWaveRows), wbytes);
        lds_dma_wait();
        if (tid < w.n) yrow[tid] = pt * (a.k + a.sh) + ps;
        if (TS != TD && shx)
            passes<TS, CHS>(a, w, T, yrow, xds[wave], row0);
        else
            passes<TD, CH>(a, w, T, yrow, xds[wave], row0);
    }
};

// -- down for the 16-pair units beside dot units -----------------------
// 64 rows per workgroup, 16 a wave.  Q8_K(h) of the unit's pairs is formed in
// LDS as the dots form it (no launch of its own), the rows come from memory with
// two super-blocks of raw bytes in flight.
template <int T, int NBH>
__device__ __forceinline__ void down_small(const BatchedArgs &a, const Unit &w, Q8L *q8h) {
    using K = Tile<T>;
    constexpr int D = 2;
    static_assert(NBH >= D, "the raw bytes' ring");
    const int wave = wave_index(), lane = threadIdx.x & 63, c = lane & 15, q = lane >> 4;
    const int row0 = blockIdx.x * kDnRows + wave * kWaveRows;
    constexpr size_t rb = (size_t)NBH * QType<T>::bytes;
    const uint8_t *W = batched_down(a, w.e) + (size_t)row0 * rb;
    const float *h = a.hbuf + (size_t)w.p0 * a.n_ff;  // the pairs' h is contiguous
    const int pc = w.p0 + min(c, w.n - 1), yr = a.ptok[pc] * (a.k + a.sh) + a.pslot[pc];
    WaveQuant<4> hq;
    hq.load(h, wave, w.n * NBH, 4);
    typename K::Raw raw[D];
#pragma unroll
    for (int i = 0; i < D; ++i) K::load(W, rb, i, raw[i]);
    hq.form<kSums32>(h, q8h, wave, w.n * NBH, 4);
    lds_barrier();
    const Q8L *x = q8h + min(c, w.n - 1) * NBH;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f}, accm[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int b = 0; b < NBH; ++b) {
        typename K::Fold f;
        K::fold(raw[b % D], f);
        if (b + D < NBH) K::load(W, rb, b + D, raw[b % D]);
        XOps xo;
        K::load_x(x[b], xo);
        xo.xd = x[b].d;
        K::step(f, xo, acc, accm);
    }
    if (c < w.n)
        *reinterpret_cast<float4 *>(a.ybuf + (size_t)yr * a.n_embd + row0 + 4 * q) =
            make_float4(acc[0] - accm[0], acc[1] - accm[1], acc[2] - accm[2], acc[3] - accm[3]);
}

// grid (n_embd / 64, max units)
template <int TD, int NBH, int TS>
__global__ __launch_bounds__(256, (TD == kTypeQ4K && NBH > 2) || (TD == kTypeQ5K && NBH > 2) ? 3 : 4) void down_dots_kernel(BatchedArgs a) {
    static_assert(kDnRows == 32 * kRowSets, "both units' rows per workgroup");
    __shared__ __align__(16) Q8L q8h[16 * NBH];
    Unit w;
    if (!load_unit(a, blockIdx.y, w)) return;
    if (TS != TD && a.sh && w.e == a.n_ids) {
        if (w.dots)
            down_dots<TS, NBH>(a, w, q8h);
        else
            down_small<TS, NBH>(a, w, q8h);
    } else {
        if (w.dots)
            down_dots<TD, NBH>(a, w, q8h);
        else
            down_small<TD, NBH>(a, w, q8h);
    }
}
// Waves a SIMD (register bound).
template <int TD, int NBH>
constexpr int kMixedWaves = TD == kTypeQ5K && NBH > 2 ? 3 : 4;
template <int TD, int NBH, int TS>
__global__ __launch_bounds__(256, (kMixedWaves<TD, NBH>)) void down_mixed_kernel(BatchedArgs a) {
    using Small = DownTile<TD, NBH, TS, 16, 1>;
    // (two chunks of Q6_K beside Q5_K rows take the registers of a fourth wave)
    using Large = DownTile<TD, NBH, TS, 32, 2, TS == TD ? 2 : 1>;
    __shared__ __align__(16) uint8_t smem[Large::kLds];
    Unit w;
    if (!load_unit(a, blockIdx.y, w)) return;
    if (w.n <= 16)
        Small::run(a, w, smem);
    else
        Large::run(a, w, smem);
}
template <int TD, int NBH, int TS>
__global__ __launch_bounds__(256, TD == kTypeQ6K ? 3 : 2) void down_large_kernel(BatchedArgs a) {
    using Large = DownTile<TD, NBH, TS, 64, 4>;
    __shared__ __align__(16) uint8_t smem[Large::kLds];
    Unit w;
    if (load_unit(a, blockIdx.y, w)) Large::run(a, w, smem);
}

template <int TG>
void launch_gateup_units(const BatchedArgs &a, hipStream_t s) {
    const dim3 gg(a.n_ff / kGuRows, a.max_units);
    if (a.units_mode == kUnitsDots)
        hipLaunchKernelGGL((gateup_dots_kernel<TG, 8, kDotGuRows>), dim3(a.n_ff / kDotGuRows, a.max_units), dim3(256), 0, s, a);
    else if (a.units_mode == kUnitsDotGateUp)
        hipLaunchKernelGGL((gateup_dots_kernel<TG, 8, kGuRows>), gg, dim3(256), 0, s, a);
    else if (a.units_mode == kUnitsMixed)
        hipLaunchKernelGGL((gateup_mixed_kernel<TG, 8>), gg, dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((gateup_large_kernel<TG, 8>), gg, dim3(256), 0, s, a);
}

template <int TD, int NBH, int TS>
void launch_down_units(const BatchedArgs &a, hipStream_t s) {
    const dim3 dg(a.n_embd / kDnRows, a.max_units);
    if (a.units_mode == kUnitsDots)
        hipLaunchKernelGGL((down_dots_kernel<TD, NBH, TS>), dg, dim3(256), 0, s, a);
    else if (a.units_mode <= kUnitsMixed)
        hipLaunchKernelGGL((down_mixed_kernel<TD, NBH, TS>), dg, dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((down_large_kernel<TD, NBH, TS>), dg, dim3(256), 0, s, a);
}

}  // namespace

hipError_t launch_expert_units(const BatchedArgs &a, hipStream_t s) {
    if (a.n_embd != 2048 || a.n_ff % kGuRows || a.n_embd % kDnRows || a.n_ff / QK > 4 || a.max_units < 1)
        return hipErrorInvalidValue;
    const int nbh = a.n_ff / QK;
    if (a.gu_type == kTypeQ4K)
        launch_gateup_units<kTypeQ4K>(a, s);
    else if (a.gu_type == kTypeQ3K)
        launch_gateup_units<kTypeQ3K>(a, s);
    else
        return hipErrorInvalidValue;
    if (a.units_mode != kUnitsDots)  // (the launch with down dots forms it)
        hipLaunchKernelGGL(pf_quant_h_kernel, dim3(a.M * (a.k + a.sh)), dim3(64 * nbh), 0, s, a);
    const int sd = a.sh ? a.sh_d_type : a.d_type;
// one set of kernels per (routed down type, super-blocks per row, shared down type)
#define HOARD_DOWN(T, N, TS)                          \
    if (a.d_type == T && nbh == N && sd == TS) {      \
        launch_down_units<T, N, TS>(a, s);            \
    } else
    HOARD_DOWN(kTypeQ6K, 3, kTypeQ6K)
    HOARD_DOWN(kTypeQ6K, 2, kTypeQ6K)
    HOARD_DOWN(kTypeQ6K, 4, kTypeQ6K)
    HOARD_DOWN(kTypeQ4K, 4, kTypeQ4K)
    HOARD_DOWN(kTypeQ4K, 3, kTypeQ4K)
    HOARD_DOWN(kTypeQ4K, 2, kTypeQ4K)
    HOARD_DOWN(kTypeQ5K, 4, kTypeQ5K)
    HOARD_DOWN(kTypeQ5K, 2, kTypeQ5K)
    HOARD_DOWN(kTypeQ5K, 2, kTypeQ6K) {
        return hipErrorInvalidValue;
    }
#undef HOARD_DOWN
    return hipGetLastError();
}

}  // namespace hoard
