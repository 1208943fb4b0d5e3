// Row dot products for K-quant rows read straight from memory: an aligned
// group of 8 lanes holds one row, its lanes an eighth of every super-block
// each, so a wave streams 8 rows.  A lane's share of a block is 16 contiguous
// quant bytes (8 for Q3_K) and the group's shares are contiguous, so the loads
// of a wave touch whole lines; the blocks ahead of the one being dotted are in
// registers (kRowAhead), where a CU holds far more bytes in flight than its
// LDS would.  Integer sums are exact (v_dot4_i32_i8, then a DPP sum over the
// group), and the fp32 block terms are added in block order, so a row's value
// is the per-block path's bit for bit.
//
// Q4_K and Q5_K blocks are 16-byte aligned; Q6_K and Q3_K blocks are only
// 2-byte aligned, which global loads take at any width.
#pragma once

#include "qblocks.h"
#include "rowdot.h"
#include "wave.h"

namespace hoard {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x2 u32x2_a2 __attribute__((aligned(2)));
typedef u32x3 u32x3_a2 __attribute__((aligned(2)));
typedef u32x4 u32x4_a2 __attribute__((aligned(2)));
typedef u32x4 u32x4_a4 __attribute__((aligned(4)));
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

// Plain loads: the lines of a block are touched by several of the wave's loads
// (header and quants, neighbouring blocks), and with the non-temporal policy
// they were fetched again (Q4_K rows 14.4 against 10.7 us for 42 MB, Q6_K rows
// 16.6 against 12.6).
template <class V>
__device__ __forceinline__ V ld_weights(const uint8_t *p) {
    return *reinterpret_cast<const V *>(p);
}

// One lane's share of a super-block of type T: load() issues its loads (the
// block at base + off, base the same in every lane of the wave, so that a step
// along the row costs scalar work only), sums() forms the lane's part of the
// block's integer sums against x.
template <int T>
struct RowShare;

// The Q4_K / Q5_K header as a lane uses it: scales of sub-blocks 2c and 2c + 1
// (c = t / 2, the 64-element chunk its quants lie in) and the min factor of
// sub-block t.
__device__ __forceinline__ void q45_header(const u32x4 &hd, int t, int &sc0, int &sc1, int &mn) {
    const bool up = t >= 4;  // sub-blocks 4..7 keep their upper two bits with 0..3
    const uint32_t sc = up ? (hd[3] & 0x0f0f0f0fu) | ((hd[1] >> 2) & 0x30303030u) : hd[1] & 0x3f3f3f3fu;
    const uint32_t mw = up ? ((hd[3] >> 4) & 0x0f0f0f0fu) | ((hd[2] >> 2) & 0x30303030u) : hd[2] & 0x3f3f3f3fu;
    const uint32_t s2 = sc >> (8 * (t & 2));
    sc0 = (int)(s2 & 0xffu);
    sc1 = (int)((s2 >> 8) & 0xffu);
    mn = (int)((mw >> (8 * (t & 3))) & 0xffu);
}
__device__ __forceinline__ int bsum_pair(const Q8L &x, int s) {  // sum of the 32 quants of sub-block s
    const uint32_t w = *reinterpret_cast<const uint32_t *>(&x.bsums[2 * s]);
    return (int)(int16_t)(w & 0xffffu) + (int)(int16_t)(w >> 16);
}

template <>
struct RowShare<kTypeQ4K> {
    u32x4 hd, q;
    __device__ __forceinline__ void load(const uint8_t *base, uint32_t off, int t) {
        hd = ld_weights<u32x4>(base + off);
        q = ld_weights<u32x4>(base + (off + (uint32_t)(16 + 16 * t)));
    }
    // Lane t covers quant bytes [16 t, 16 t + 16): 16 elements of sub-block
    // 2 (t / 2) in the low nibbles, of 2 (t / 2) + 1 in the high ones.
    __device__ __forceinline__ void sums(const Q8L &x, int t, int &isum, int &msum) const {
        const int c = t >> 1, h = t & 1;
        const u32x4 xl = *reinterpret_cast<const u32x4 *>(&x.qs[16 * c + 4 * h]);
        const u32x4 xh = *reinterpret_cast<const u32x4 *>(&x.qs[16 * c + 8 + 4 * h]);
        int lo = 0, hi = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            lo = sdot4(q[k] & 0x0f0f0f0fu, xl[k], lo);
            hi = sdot4((q[k] >> 4) & 0x0f0f0f0fu, xh[k], hi);
        }
        int sc0, sc1, mn;
        q45_header(hd, t, sc0, sc1, mn);
        isum = sc0 * lo + sc1 * hi;
        msum = mn * bsum_pair(x, t);
    }
    __device__ __forceinline__ float d() const { return half_bits_to_float(hd[0] & 0xffffu); }
    __device__ __forceinline__ float dmin() const { return half_bits_to_float(hd[0] >> 16); }
};

template <>
struct RowShare<kTypeQ5K> {
    u32x4 hd, qh, q;
    __device__ __forceinline__ void load(const uint8_t *base, uint32_t off, int t) {
        hd = ld_weights<u32x4>(base + off);
        qh = ld_weights<u32x4>(base + (off + (uint32_t)(16 + 16 * (t & 1))));
        q = ld_weights<u32x4>(base + (off + (uint32_t)(48 + 16 * t)));
    }
    // Q4_K's share with the fifth bits: bit 2c / 2c + 1 of the qh byte of the
    // same position for the low / high nibbles.
    __device__ __forceinline__ void sums(const Q8L &x, int t, int &isum, int &msum) const {
        const int c = t >> 1, h = t & 1;
        const u32x4 xl = *reinterpret_cast<const u32x4 *>(&x.qs[16 * c + 4 * h]);
        const u32x4 xh = *reinterpret_cast<const u32x4 *>(&x.qs[16 * c + 8 + 4 * h]);
        int lo = 0, hi = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t b = qh[k] >> (2 * c);
            lo = sdot4((q[k] & 0x0f0f0f0fu) | ((b & 0x01010101u) << 4), xl[k], lo);
            hi = sdot4(((q[k] >> 4) & 0x0f0f0f0fu) | ((b & 0x02020202u) << 3), xh[k], hi);
        }
        int sc0, sc1, mn;
        q45_header(hd, t, sc0, sc1, mn);
        isum = sc0 * lo + sc1 * hi;
        msum = mn * bsum_pair(x, t);
    }
    __device__ __forceinline__ float d() const { return half_bits_to_float(hd[0] & 0xffffu); }
    __device__ __forceinline__ float dmin() const { return half_bits_to_float(hd[0] >> 16); }
};

template <>
struct RowShare<kTypeQ6K> {
    u32x4 ql, qh;
    u32x2 sc;
    uint16_t db;
    __device__ __forceinline__ void load(const uint8_t *base, uint32_t off, int t) {
        ql = ld_weights<u32x4_a2>(base + (off + (uint32_t)(16 * t)));
        qh = ld_weights<u32x4_a2>(base + (off + (uint32_t)(128 + 32 * (t >> 2) + 16 * (t & 1))));
        sc = ld_weights<u32x2_a2>(base + (off + (uint32_t)(192 + 8 * (t >> 2))));
        db = ld_weights<uint16_t>(base + (off + (uint32_t)(208)));
    }
    // Lane t covers ql bytes [16 t, 16 t + 16): in half n = t / 4, with
    // i = t & 3, the 16 elements of scale group 8 n + i (low nibbles, qh bits
    // 2 (i / 2)) and of group 8 n + 4 + i (high nibbles, 4 bits further up).
    __device__ __forceinline__ void sums(const Q8L &x, int t, int &isum, int &msum) const {
        const int g = 8 * (t >> 2) + (t & 3), sh = t & 2;
        const u32x4 xl = *reinterpret_cast<const u32x4 *>(&x.qs[4 * g]);
        const u32x4 xh = *reinterpret_cast<const u32x4 *>(&x.qs[4 * g + 16]);
        int lo = 0, hi = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t b = qh[k] >> sh;
            lo = sdot4((q_lo(k)) | ((b & 0x03030303u) << 4), xl[k], lo);
            hi = sdot4((q_hi(k)) | (b & 0x30303030u), xh[k], hi);
        }
        const int s0 = (int)(int8_t)(sc[0] >> (8 * (t & 3))), s1 = (int)(int8_t)(sc[1] >> (8 * (t & 3)));
        isum = s0 * (lo - 32 * (int)x.bsums[g]) + s1 * (hi - 32 * (int)x.bsums[g + 4]);
        msum = 0;
    }
    __device__ __forceinline__ uint32_t q_lo(int k) const { return ql[k] & 0x0f0f0f0fu; }
    __device__ __forceinline__ uint32_t q_hi(int k) const { return (ql[k] >> 4) & 0x0f0f0f0fu; }
    __device__ __forceinline__ float d() const { return half_bits_to_float(db); }
    __device__ __forceinline__ float dmin() const { return 0.0f; }
};

template <>
struct RowShare<kTypeQ3K> {
    u32x2 q, hm;
    u32x3 sc;
    uint16_t db;
    __device__ __forceinline__ void load(const uint8_t *base, uint32_t off, int t) {
        q = ld_weights<u32x2_a2>(base + (off + (uint32_t)(32 + 8 * t)));
        hm = ld_weights<u32x2_a2>(base + (off + (uint32_t)(8 * (t & 3))));
        sc = ld_weights<u32x3_a2>(base + (off + (uint32_t)(96)));
        db = ld_weights<uint16_t>(base + (off + (uint32_t)(108)));
    }
    // Lane t covers qs bytes [8 t, 8 t + 8): in half n = t / 4 the elements
    // 128 n + 32 j + 8 (t & 3) + 0..7, j = 0..3, half of scale group
    // 8 n + 2 j + ((t & 3) / 2); the even lane of the pair that shares the
    // group takes its -4 * bsum.
    __device__ __forceinline__ void sums(const Q8L &x, int t, int &isum, int &msum) const {
        const int n = t >> 2, i = t & 3;
        isum = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const u32x2 xw = *reinterpret_cast<const u32x2 *>(&x.qs[32 * n + 8 * j + 2 * i]);
            int s = 0;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const uint32_t h = (hm[k] >> (4 * n + j)) & 0x01010101u;
                s = sdot4(((q[k] >> (2 * j)) & 0x03030303u) | (h << 2), xw[k], s);
            }
            const int g = 8 * n + 2 * j + (i >> 1);
            const int corr = (t & 1) ? 0 : 4 * (int)x.bsums[g];
            // scale g: low nibble from byte g % 8, shifted by 4 for g >= 8; upper two bits
            // from byte 8 + g % 4, bits 2 (g / 4); g / 4 = 2 n + j / 2
            const uint32_t lw = j & 2 ? sc[1] : sc[0];
            const int b = 8 * (2 * (j & 1) + (i >> 1));
            const int lo = (int)((lw >> (b + 4 * n)) & 0x0fu);
            const int hi = (int)((sc[2] >> (b + 2 * (2 * n + (j >> 1)))) & 3u);
            isum += ((lo | (hi << 4)) - 32) * (s - corr);
        }
        msum = 0;
    }
    __device__ __forceinline__ float d() const { return half_bits_to_float(db); }
    __device__ __forceinline__ float dmin() const { return 0.0f; }
};

// Blocks of a row a lane holds in flight while it dots the ones before them:
// 4 where a block is two 16-byte loads, 3 where it takes more.  Deeper rings
// cost waves in flight (registers): at 8 experts of 4096 x 1536 a Q6_K down
// launch took 15.3 us at 2, 15.5 at 3, 17.8 at 4, a Q4_K gate/up launch 16.4,
// 16.7 and 15.7.
template <int T>
constexpr int kRowAhead = T == kTypeQ4K ? 4 : 3;

// The rows a wave's 8-lane groups stream, one a group, at base + off (base
// wave-uniform): begin() issues the first kAhead blocks' loads, finish()
// dots them while the later ones fly.  A round's loads past the row's last
// block repeat that block, so every round but the last issues the same loads.
// Every lane of the group returns the row's value.
template <int T>
struct RowStream {
    static constexpr int kAhead = kRowAhead<T>;
    RowShare<T> s[kAhead];
    __device__ __forceinline__ void load(int i, const uint8_t *base, uint32_t off, int b, int nb, int t) {
        s[i].load(base + (size_t)(b < nb ? b : nb - 1) * QType<T>::bytes, off, t);
    }
    __device__ __forceinline__ void begin(const uint8_t *base, uint32_t off, int nb, int t) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i) load(i, base, off, i, nb, t);
    }
    __device__ __forceinline__ void step(int i, const Q8L &x, int t, float &acc, float &accm) {
        int isum, msum;
        s[i].sums(x, t, isum, msum);
        isum = group8_sum(isum);
        acc = acc + (s[i].d() * x.d) * (float)isum;
        if constexpr (QType<T>::has_min) accm = accm + (s[i].dmin() * x.d) * (float)group8_sum(msum);
    }
    __device__ __forceinline__ float finish(const uint8_t *base, uint32_t off, const Q8L *x, int nb, int t) {
        float acc = 0.0f, accm = 0.0f;
        int b0 = 0;
#pragma unroll 1
        for (; b0 + kAhead < nb; b0 += kAhead) {
#pragma unroll
            for (int i = 0; i < kAhead; ++i) {
                step(i, x[b0 + i], t, acc, accm);
                __builtin_amdgcn_sched_barrier(0);
                load(i, base, off, b0 + i + kAhead, nb, t);
            }
        }
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            if (b0 + i < nb) step(i, x[b0 + i], t, acc, accm);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (QType<T>::has_min)
            return acc - accm;
        else
            return acc;
    }
};

// Q8_K of blocks first, first + step, ... below end of x into q, by one wave.
// load() issues the loads of the first K blocks; the rest are loaded one by
// one as the blocks are formed (behind whatever the wave loaded in between).
// One quantiser in a loop that shifts the loaded blocks down: unrolled K
// times it was most of a kernel's code.  x is 4-byte aligned.
template <int K>
struct WaveQuant {
    f32x4_a4 v[K];
    __device__ __forceinline__ void load(const float *x, int first, int end, int step) {
#pragma unroll
        for (int i = 0; i < K; ++i) get(i, x, min(first + i * step, end - 1));
    }
    __device__ __forceinline__ void get(int i, const float *x, int b) {
        v[i] = *reinterpret_cast<const f32x4_a4 *>(x + (size_t)b * QK + 4 * (threadIdx.x & 63));
    }
    template <int Sums = kSumsInt>
    __device__ __forceinline__ void form(const float *x, Q8L *q, int first, int end, int step) {
#pragma unroll 1
        for (int b = first; b < end; b += step) {
            const float w[4] = {v[0][0], v[0][1], v[0][2], v[0][3]};
#pragma unroll
            for (int i = 0; i + 1 < K; ++i) v[i] = v[i + 1];
            if (b + K * step < end) get(K - 1, x, b + K * step);
            wave_quantize_q8l_regs<Sums>(w, q + b);
        }
    }
};

}  // namespace hoard
