// Work units of a batch, and the expert products of those that hold few pairs:
// at most kDotTokens of them computed token by token with the per-token row
// dots, which give the single-token path's bits.  The larger units run on the
// int8 MFMA bodies of prefill.hip, in the same launches.
#pragma once

#include "kernels.h"
#include "lds_dma.h"
#include "qblocks.h"
#include "rowdot.h"
#include "rowstream.h"
#include "wave.h"

namespace hoard {

// A work unit: expert e, its pairs [p0, p0 + n) in sorted order, whether it is a
// dot unit and then its pairs' tokens, a byte each; one 16-byte record (a place
// past the last unit holds n = 0), so a workgroup knows its work after one memory
// latency.
struct Unit {
    int e, p0, n;
    bool dots;
    uint32_t tok;
};
__device__ __forceinline__ bool load_unit(const BatchedArgs &a, int unit, Unit &w) {
    const int4 r = *reinterpret_cast<const int4 *>(a.units + 4 * unit);
    w.e = r.x;
    w.p0 = r.y;
    w.n = r.z & 0xffff;
    w.dots = r.z & kDotUnit;
    w.tok = (uint32_t)r.w;
    return w.n > 0;
}

// Gather the Q8_K row (nb blocks) of token tt into LDS at xs, 16-byte granules
// spread over the workgroup's nw waves (issued, not waited for).
template <int NBX>
__device__ __forceinline__ void gather_token(uint8_t *xs, const uint8_t *q8base, int tt, int wave, int nw) {
    constexpr int kTokGran = NBX * (int)sizeof(Q8L) / 16;
    const int lane = threadIdx.x & 63;
    for (int k = wave; 64 * k < kTokGran; k += nw) {
        const int p = 64 * k + lane;
        if (p < kTokGran) dma_lanes(xs + 1024 * k, q8base + (size_t)tt * (NBX * sizeof(Q8L)) + 16 * p);
    }
}

// -- gate/up: 16 rows of gate (waves 0, 1) and of up (waves 2, 3) from row0 on --
// One 8-lane group per row, lane t holding the token's Q8_K block t; the weight
// tile is contiguous rows, copied into LDS in one burst.  x goes into LDS with
// the tile, a token at a time (a vector load issued during the compute would
// queue behind the tile copies of the other workgroups on this CU).
// A larger group is cut into several units (its weights are then read again,
// from the caches), so that no workgroup is left with a long chain of tokens.
constexpr int kDotGuRows = 16;
template <int TGU, int NB>
struct DotGateUp {
    static_assert(NB == 8, "one 8-lane group per row, one lane per super-block");
    static_assert(TGU == kTypeQ4K || TGU == kTypeQ3K, "gate/up rows are Q4_K or Q3_K");
    static constexpr int kRowBytes = NB * QType<TGU>::bytes;
    static constexpr int kTileBytes = 8 * kRowBytes;  // a wave's rows
    static_assert(kTileBytes % 16 == 0, "the tile copies in 16-byte units");
    static constexpr int kXBytes = NB * (int)sizeof(Q8L);
    // LDS: the four waves' tiles, one token's x, the gate and up values
    static constexpr int kLds = 4 * kTileBytes + kXBytes + 2 * kDotGuRows * kDotTokens * (int)sizeof(float);

    static __device__ __forceinline__ void run(const BatchedArgs &a, const Unit &w, int row0, uint8_t *smem) {
        const int wave = wave_index(), lane = threadIdx.x & 63, t8 = lane & 7, grp = lane >> 3;
        const int up = wave >> 1, r8 = 8 * (wave & 1);
        uint8_t *wt = smem + wave * kTileBytes, *xs = smem + 4 * kTileBytes;
        float *gu = reinterpret_cast<float *>(xs + kXBytes);  // [2][kDotGuRows][kDotTokens]
        const uint8_t *W = (up ? batched_up(a, w.e) : batched_gate(a, w.e)) + (size_t)(row0 + r8) * kRowBytes;
        const Q8L *xl = reinterpret_cast<const Q8L *>(xs);
        for (int c = 0; c < w.n; ++c) {
            if (c > 0) __syncthreads();  // every wave is done with the previous token
            gather_token<NB>(xs, a.q8x, (int)((w.tok >> (8 * c)) & 0xffu), wave, 4);
            if (c == 0) dma_wave_copy_nt(wt, W, kTileBytes);
            lds_dma_wait();
            __syncthreads();
            const uint8_t *rp = wt + grp * kRowBytes;
            float v;
            if constexpr (TGU == kTypeQ3K)
                v = lpb_row_q3k_mem<NB, true>(rp, xl[t8], t8);
            else
                v = lpb_row_q4k_mem<NB, true>(rp, xl[t8], t8);
            if (t8 == NB - 1) gu[(up * kDotGuRows + r8 + grp) * kDotTokens + c] = v;
        }
        __syncthreads();
        // h = silu(gate) * up
        const int r = threadIdx.x % kDotGuRows, c = threadIdx.x / kDotGuRows;
        if (c < w.n) {
            const float g = gu[r * kDotTokens + c], uu = gu[(kDotGuRows + r) * kDotTokens + c];
            a.hbuf[(size_t)(w.p0 + c) * a.n_ff + row0 + r] = g / (1.0f + expf(-g)) * uu;
        }
    }
};

// -- down: rows of the unit's expert, y to its (token, slot) place -------------
// 32 kRowSets rows per workgroup of four waves: a wave's rows (kRowSets an 8-lane
// group) go from memory to registers whole, all their blocks in flight at once,
// while the workgroup forms Q8_K(h) of the unit's pairs in LDS from h (a launch
// of its own for that takes 4 to 5 us); then each pair's dots from the registers.
// Bound by the weight stream's latency at few tokens, by the dots and the forming
// at 16 (waves ready but not issued for 54 % of their cycles): Qwen3-30B at 4
// tokens 10.7 us a launch, 16.4 with the tile in LDS, one wave a workgroup and
// Q8_K(h) in a launch before it; at 16 tokens 28.4 against 27.7 and 4.9.
constexpr int kRowSets = 2;  // row sets of 8 a wave takes of the down rows (four of the shortest rows measured slower)
template <int T, int NBH>
__device__ __forceinline__ void down_dots(const BatchedArgs &a, const Unit &w, Q8L *q8h) {
    const int wave = wave_index(), lane = threadIdx.x & 63, t8 = lane & 7, grp = lane >> 3;
    constexpr int RS = kRowSets;
    const int row0 = (blockIdx.x * 4 + wave) * 8 * RS;
    const float *h = a.hbuf + (size_t)w.p0 * a.n_ff;  // the pairs' h is contiguous
    int slot[kDotTokens];
#pragma unroll
    for (int c = 0; c < kDotTokens; ++c) slot[c] = a.pslot[w.p0 + min(c, w.n - 1)];
    WaveQuant<NBH> hq;  // a wave forms at most NBH of the kDotTokens * NBH blocks
    hq.load(h, wave, w.n * NBH, 4);
    RowShare<T> s[RS][NBH];
    const uint8_t *base = batched_down(a, w.e) + (size_t)row0 * (NBH * QType<T>::bytes);
#pragma unroll
    for (int p = 0; p < RS; ++p)
#pragma unroll
        for (int b = 0; b < NBH; ++b)
            s[p][b].load(base + b * QType<T>::bytes, (uint32_t)((8 * p + grp) * (NBH * QType<T>::bytes)), t8);
    hq.form(h, q8h, wave, w.n * NBH, 4);
    lds_barrier();
    const int kk = a.k + a.sh;  // output slots per token
    for (int c = 0; c < w.n; ++c) {
        const Q8L *x = q8h + c * NBH;
        float v = 0.0f;  // lane t of a group keeps row set t's value
#pragma unroll
        for (int p = 0; p < RS; ++p) {
            float acc = 0.0f, accm = 0.0f;
#pragma unroll
            for (int b = 0; b < NBH; ++b) {
                int isum, msum;
                s[p][b].sums(x[b], t8, isum, msum);
                isum = group8_sum(isum);
                acc = acc + (s[p][b].d() * x[b].d) * (float)isum;
                if constexpr (QType<T>::has_min) accm = accm + (s[p][b].dmin() * x[b].d) * (float)group8_sum(msum);
                __builtin_amdgcn_sched_barrier(0);  // a block's operands at a time
            }
            const float r = QType<T>::has_min ? acc - accm : acc;
            v = t8 == p ? r : v;
        }
        const int sl = c == 0 ? slot[0] : c == 1 ? slot[1] : c == 2 ? slot[2] : slot[3];
        float *y = a.ybuf + ((size_t)((w.tok >> (8 * c)) & 0xffu) * kk + sl) * a.n_embd + row0;
        if (t8 < RS) y[8 * t8 + grp] = v;
    }
}

}  // namespace hoard
