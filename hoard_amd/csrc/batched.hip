// Batched expert stage for M tokens (speculative verify / prefill): routing,
// grouping by expert into work units, so that every selected expert's weights
// are read once per unit, and the combine.
//
// Counterpart of ggml_mul_mat_id over the slot pool with per-token ids
// (src/run_specloop.cpp:126-139; all-resident form src/run_m1.cpp:97-108)
// followed by the weighted sum over the selected experts.
//
// The expert products are in prefill.hip: units of a few pairs on per-token
// dots, larger ones on int8 MFMA.
#include "kernels.h"
#include "lds_dma.h"
#include "qblocks.h"
#include "rowdot.h"
#include "router_tail.h"

namespace hoard {

namespace {

constexpr int kMaxExperts = 1024;
constexpr int kMaxTok = kBatchedMaxTokens;  // tokens of a verify-sized batch
static_assert(kDotTokens == 4 && kMaxDotTokens <= 256, "a unit's tokens are the bytes of one word");
static_assert(kMaxDotTokens / 32 * (kMaxExperts + 1) <= 8448, "their grouping takes the one-pass form");
static_assert(sizeof(Q8L) == kQ8LBytes, "Q8_K block size shared with the host");

__device__ __forceinline__ Q8L *q8(uint8_t *p) { return reinterpret_cast<Q8L *>(p); }

// -- route: router logits, softmax / top-k, Q8_K of fx, grouping by expert ----
// One launch replaces the router kernels and the grouping pass.  A workgroup
// (4 waves) takes R router rows against kRouteTok tokens, a wave per token and
// a half-wave per row at a time, with the single-token router's per-row
// accumulation order (lane l of 32 owns elements l, l+32, ...; ggml's f32 dot
// fold).  Up to 8 tokens two rows per workgroup, above that four (fewer
// copies of the tokens' fx): measured per layer, four rows against two took
// 0.5 us off at 16 tokens and 2.8 at 32 (Qwen3-30B shape), 3.3 and 7.5 with
// 512 experts (Qwen3-Next), and added 1.2 us at 4 tokens; eight rows were
// slower than four everywhere.  A remainder of one row (a shared expert's
// gate row after a multiple of R routed rows) goes to the last workgroup of
// the row range as an extra pass instead of a workgroup of its own: with 512
// experts and four token groups the extra workgroups would not fit the two a
// CU that the LDS allows, and a second round of workgroups would follow the
// first.  The last
// workgroup of a token group (device-scope counter) runs the tails of its
// tokens; the last token group's tail workgroup then groups the (token, slot)
// pairs by expert.  Waves with a spare slot quantise fx to Q8_K.
constexpr int kRouteTok = 4;
constexpr int kRouteN = 2048;  // n_embd of the batched path

// Group the (token, slot) pairs by expert (all threads of the workgroup call
// this).  A token selects an expert at most once, so a per-expert bitmask of
// tokens orders each group by token; groups are numbered in ascending expert
// id.
// With caller ids (ysrc, bad: the grouping workgroup's LDS copies) a pair that
// repeats an earlier id of its token, or whose token has an id out of range,
// joins no group.
__device__ __forceinline__ bool pair_computed(const BatchedArgs &a, const int *ysrc, const int *bad, int p) {
    return !ysrc || (ysrc[p] == p % a.k && !bad[p / a.k]);
}

// LDS of the grouping passes; the route kernel lays it over its staging
// buffers, which are free by then.
struct GroupLds {
    unsigned mask[kMaxExperts];  // tokens (of a chunk) selecting each expert
    unsigned cnt[kMaxExperts];   // pairs per expert
    int base[kMaxExperts];       // next sorted position of each expert
    int ubase[kMaxExperts];      // first unit of each expert
    int total;
};

__device__ void group_units(const BatchedArgs &a, GroupLds &g);

// Token t, the c-th of expert e's group, into its unit's record where the group
// is cut into dot units.
__device__ __forceinline__ void unit_token(const BatchedArgs &a, const GroupLds &g, int e, int c, int t) {
    if (a.units_mode <= kUnitsDotGateUp && g.cnt[e] < kMfmaPairs)
        reinterpret_cast<uint8_t *>(a.units + 4 * (g.ubase[e] + c / kDotTokens) + 3)[c % kDotTokens] = (uint8_t)t;
}

// Grouping of a batch of at most 32 tokens (all threads of the workgroup): a
// group's mask gives its size and each pair's place.  sel: the pairs' selected
// experts, in LDS.  Dot units carry their tokens in the record.
__device__ void group_by_expert(const BatchedArgs &a, GroupLds &g, const int *sel, const int *ysrc = nullptr,
                                const int *bad = nullptr) {
    unsigned *mask = g.mask;
    const int tid = threadIdx.x, nt = blockDim.x, E = a.n_ids, P = a.M * a.k;
    for (int e = tid; e < E; e += nt) mask[e] = 0u;
    if (a.sh && tid == 0) mask[E] = a.M < 32 ? (1u << a.M) - 1u : ~0u;  // the shared expert: every token
    __syncthreads();
    // out-of-range selections count as expert 0
    auto expert = [&](int p) { return sel[p] < 0 || sel[p] >= E ? 0 : sel[p]; };
    for (int p = tid; p < P; p += nt)
        if (pair_computed(a, ysrc, bad, p)) atomicOr(&mask[expert(p)], 1u << (p / a.k));
    __syncthreads();
    for (int e = tid; e < E + a.sh; e += nt) g.cnt[e] = (unsigned)__popc(mask[e]);
    __syncthreads();
    if (tid < 64) group_units(a, g);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the records are written before their token bytes
    __syncthreads();
    const int kk = a.k + a.sh;
    for (int p = tid; p < a.M * kk; p += nt) {
        const int t = p / kk, j = p - t * kk;
        int e = E;
        if (j < a.k) {
            if (!pair_computed(a, ysrc, bad, t * a.k + j)) continue;
            e = expert(t * a.k + j);
        }
        const int c = __popc(mask[e] & ((1u << t) - 1u));
        a.ptok[g.base[e] + c] = t;
        a.pslot[g.base[e] + c] = j;
        unit_token(a, g, e, c, t);
    }
}

// Groups in ascending expert order and their units from the per-expert pair
// counts g.cnt (wave 0 of the grouping workgroup): hist, the unit records {expert,
// first sorted pair, pairs, 0} (every place past the last unit zeroed),
// n_unique, and g.base[e] / g.ubase[e], the first sorted place and
// the first unit of expert e.  The shared expert's units, which hold the most
// pairs and take longest, come first: at the end they outlast the rest (512
// experts, 16 tokens 68 us/layer, 61 so; 256 experts 57 and 51).
__device__ void group_units(const BatchedArgs &a, GroupLds &g) {
    const int tid = threadIdx.x, E = a.n_ids + a.sh;
    {
        // groups and units in ascending expert order: lane owns a contiguous run of experts
        const int lane = tid, per = (E + 63) / 64, e0 = lane * per;
        int cg = 0, cu = 0, cp = 0;
        for (int e = e0; e < e0 + per && e < E; ++e) {
            const int c = (int)g.cnt[e];
            cg += c ? 1 : 0;
            const int us = unit_shift(a.units_mode, c);
            cu += (c + (1 << us) - 1) >> us;
            cp += c;
        }
        int ig = cg, iu = cu, ip = cp;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int og = __shfl_up(ig, off), ou = __shfl_up(iu, off), op = __shfl_up(ip, off);
            if (lane >= off) {
                ig += og;
                iu += ou;
                ip += op;
            }
        }
        const int us = a.sh ? unit_shift(a.units_mode, (int)g.cnt[E - 1]) : 0;
        const int shu = a.sh ? ((int)g.cnt[E - 1] + (1 << us) - 1) >> us : 0;
        int ui = shu + iu - cu, pi = ip - cp;
        for (int e = e0; e < e0 + per && e < E; ++e) {
            const int c = (int)g.cnt[e];
            if (e == a.n_ids) ui = 0;
            a.hist[e] = (unsigned)c;
            g.base[e] = pi;
            g.ubase[e] = ui;
            const int u = 1 << unit_shift(a.units_mode, c), flag = u == kDotTokens ? kDotUnit : 0;
            for (int s0 = 0; s0 < c; s0 += u, ++ui)
                *reinterpret_cast<int4 *>(a.units + 4 * ui) = make_int4(e, pi + s0, min(u, c - s0) | flag, 0);
            pi += c;
        }
        if (lane == 63) {
            a.n_unique[0] = ig - a.sh;  // routed experts used
            g.total = ip;  // pairs in all groups
        }
        // the grid's unit places past the last unit hold no pairs, so a workgroup
        // learns from its own place alone whether it has work
        for (int x = __shfl(iu, 63) + lane; x < a.max_units; x += 64)
            *reinterpret_cast<int4 *>(a.units + 4 * x) = make_int4(0, 0, 0, 0);
    }
}

// Grouping of a prefill-sized batch (all threads of one workgroup): the
// computed (token, slot) pairs sorted by (expert, token) into ptok / pslot, the
// groups (used experts in ascending order) and the work
// units (of one group each).  pe[p] (in LDS) is the
// expert of pair p, or -1 for a pair that joins no group.  The order within an
// expert comes from chunks of at most 32 tokens taken in token order: a pair's
// place is its expert's running base plus the tokens of its chunk before it
// that select the same expert (a token joins a group at most once).
__device__ void group_large(const BatchedArgs &a, GroupLds &g, const int *pe, int *sorted) {
    const int tid = threadIdx.x, nt = blockDim.x, E = a.n_ids + a.sh, k = a.k + a.sh, P = a.M * k;
    for (int e = tid; e < E; e += nt) g.cnt[e] = 0u;
    __syncthreads();
    for (int p = tid; p < P; p += nt)
        if (pe[p] >= 0) atomicAdd(&g.cnt[pe[p]], 1u);
    __syncthreads();
    if (tid < 64) group_units(a, g);
    __syncthreads();
    const int tpc = min(32, max(1, nt / k));  // tokens per chunk: one mask bit each
    for (int t0 = 0; t0 < a.M; t0 += tpc) {
        for (int e = tid; e < E; e += nt) g.mask[e] = 0u;
        __syncthreads();
        const int pend = min(P, (t0 + tpc) * k);
        for (int p = t0 * k + tid; p < pend; p += nt)
            if (pe[p] >= 0) atomicOr(&g.mask[pe[p]], 1u << (p / k - t0));
        __syncthreads();
        for (int p = t0 * k + tid; p < pend; p += nt) {
            const int e = pe[p];
            if (e < 0) continue;
            const int t = p / k;
            const int pos = g.base[e] + __popc(g.mask[e] & ((1u << (t - t0)) - 1u));
            sorted[pos] = t | (p - t * k) << 16;
        }
        __syncthreads();
        for (int e = tid; e < E; e += nt) g.base[e] += __popc(g.mask[e]);
        __syncthreads();
    }
}

// Q8_K of a block of fx with the sums the expert kernels of this call read.
__device__ __forceinline__ void quantize_x(const BatchedArgs &a, const float *x, Q8L *out) {
    if (a.units_mode > kUnitsDotGateUp && a.gu_type == kTypeQ3K)
        wave_quantize_q8l<kSums16>(x, out);
    else if (a.units_mode > kUnitsDotGateUp)
        wave_quantize_q8l<kSums32>(x, out);
    else
        wave_quantize_q8l(x, out);
}

template <int R>
__global__ __launch_bounds__(256) void route_kernel(BatchedArgs a) {
    constexpr int n = kRouteN, nb = kRouteN / QK;
    const int E = a.E;
    const int wave = wave_index(), lane = threadIdx.x & 63, l = lane & 31;
    const int tg = blockIdx.y;
    const int t = tg * kRouteTok + wave;  // this wave's token; its half-waves take one row each
    // rows 0..E-1 are the router's; row E (with a shared expert) is its gate row
    const int r0 = blockIdx.x * R;
    const int nrows = blockIdx.x == gridDim.x - 1 ? E + a.sh - r0 : R;  // R + 1 with a one-row remainder
    // the workgroup's token rows and router rows go to LDS in one burst, so
    // that every load is in flight at once; the dot then reads them in the
    // per-lane order the accumulation needs
    __shared__ __align__(16) float xl[kRouteTok][kRouteN];
    __shared__ __align__(16) float wl[R + 1][kRouteN];
    if (t < a.M) dma_wave_copy(reinterpret_cast<uint8_t *>(xl[wave]), reinterpret_cast<const uint8_t *>(a.fx + (size_t)t * n),
                               n * (int)sizeof(float));
    {
        // the rows' 1 KB pieces, dealt to the four waves in turn
        constexpr int kPieces = n * (int)sizeof(float) / 1024;
        for (int c = wave; c < nrows * kPieces; c += 4) {
            const int rr = c / kPieces, o = (c % kPieces) * 1024;
            const float *src = r0 + rr < E ? a.router + (size_t)(r0 + rr) * n : a.sh_gate_inp;
            dma_chunk(reinterpret_cast<uint8_t *>(wl[rr]) + o, reinterpret_cast<const uint8_t *>(src) + o);
        }
    }
    lds_dma_wait();
    __syncthreads();
    if (t < a.M) {
        const float *x = xl[wave];
        // half-wave h takes rows rp + h, rp = 0, 2, ...; the R / 2 rows of a lane
        // accumulate side by side, so their FMA chains overlap
        static_assert(R % 2 == 0, "two rows a pass, one a half-wave");
        constexpr int kP = R / 2;
        const float *wr[kP];
        float acc[kP];
#pragma unroll
        for (int j = 0; j < kP; ++j) {
            wr[j] = wl[min(2 * j + (lane >> 5), nrows - 1)];
            acc[j] = 0.0f;
        }
#pragma unroll 8
        for (int i = 0; i < n; i += 32) {
            const float xv = x[i + l];
#pragma unroll
            for (int j = 0; j < kP; ++j) acc[j] = fmaf(wr[j][i + l], xv, acc[j]);
        }
        // the remainder row, on both half-waves (the second one's result is
        // past the rows and not stored)
        float acc_r = 0.0f;
        if (nrows > R) {
            const float *w = wl[R];
#pragma unroll 8
            for (int i = 0; i < n; i += 32) acc_r = fmaf(w[i + l], x[i + l], acc_r);
        }
#pragma unroll
        for (int j = 0; j <= kP; ++j) {
            if (j == kP && nrows <= R) break;
            float v = j < kP ? acc[j] : acc_r;
            v = v + __shfl_xor(v, 16);
            v = v + __shfl_xor(v, 8);
            v = v + __shfl_xor(v, 4);
            v = v + __shfl_xor(v, 1);
            v = v + __shfl_xor(v, 2);
            const int row = r0 + 2 * j + (lane >> 5);
            if (l == 0 && row < E)
                __hip_atomic_store(a.logits + (size_t)t * E + row, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            else if (l == 0 && row == E && a.sh)
                a.sgl[t] = v;
        }
        // Q8_K of fx: workgroup i of a token group quantises blocks i, i + gridDim.x, ...
        // of its tokens, so every block is formed whatever the expert count (grid width)
        for (int b = blockIdx.x; b < nb; b += gridDim.x) quantize_x(a, x + b * QK, q8(a.q8x) + (size_t)t * nb + b);
    }
    // Completion protocol without cache-flushing fences: the logits and the
    // tails' sel / wsel are stored at device scope (through to memory, past
    // the per-XCD L2) and read back at device scope; each wave waits for its
    // stores to be acknowledged before its workgroup counts itself done.
    __shared__ int last;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0)
        last = __hip_atomic_fetch_add(&a.counters[tg], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
               gridDim.x - 1;
    __syncthreads();
    if (!last) return;
    // the selections of every token, in LDS over the staging buffers, which are free
    static_assert(sizeof(GroupLds) <= sizeof(xl) && sizeof(int) * kMaxTok * kMaxK <= sizeof(wl), "grouping LDS");
    int *sel_s = reinterpret_cast<int *>(&wl[0][0]);
    const bool one = gridDim.y == 1;  // one token group: this workgroup holds every selection
    for (int tt = wave; tt < kRouteTok; tt += 4) {
        const int tok = tg * kRouteTok + tt;
        if (tok < a.M) {
            const int id = router_tail<true>(a.logits, E, a.k, a.renorm, a.sel, a.wsel, tok);
            if (one && lane < a.k) sel_s[tok * a.k + lane] = id;
        }
    }
    if (threadIdx.x == 0) __hip_atomic_store(&a.counters[tg], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (!one) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0)
            last = __hip_atomic_fetch_add(&a.counters[kBatchedCounters - 1], 1u, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT) == gridDim.y - 1;
        __syncthreads();
        if (!last) return;
        for (int p = threadIdx.x; p < a.M * a.k; p += blockDim.x)
            sel_s[p] = __hip_atomic_load(a.sel + p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (threadIdx.x == 0)
            __hip_atomic_store(&a.counters[kBatchedCounters - 1], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    group_by_expert(a, *reinterpret_cast<GroupLds *>(&xl[0][0]), sel_s);
}

// -- prefill-sized routing: tiled router GEMM, then tails, then the grouping -----
// Logits of 16 experts x TT tokens per workgroup of 512 threads (TT = 16, or 8
// where 16-token tiles would leave CUs idle).  Thread (group q = tid / 32, lane
// l = tid % 32) holds accumulator l of ggml's x86 f32 dot (elements 32 i + l,
// i ascending) for 4 experts x TT / 4 tokens: the rows and tokens pass through
// LDS 512 elements at a time, 8 (6) reads for every 16 (8) dots.  The 32
// accumulators of a dot sit in the 32 lanes of a half-wave, which fold them in
// ggml's order, so every logit is the single-token router's.
// One workgroup per CU: eight waves (two per SIMD) took 4 us less per launch
// than four waves with 4 x 8 dots each, sixteen waves with 2 x 4 each 1 us
// more than eight.  Each K step costs a wait and a barrier besides its dots:
// 512-element steps (4 of them) took 3.5 us less per launch than 256-element
// ones (8), and 1024-element ones without a second buffer 1.6 us more than
// 512 at M = 512 (four waves).  8-token tiles where 16-token ones would fill
// at most half the CUs: 2.5 us less per layer at 128 tokens of 128 experts
// (2.2 more at 512, where 16-token tiles fill the CUs once).
constexpr int kTileE = 16;

// K steps in LDS: the current one and the next in flight (four buffers, three
// steps in flight, measured the same: once one step is prefetched the dots and
// the per-step barrier set the pace).  kTileK = 512: 128 KB of LDS, one
// workgroup per CU; 256: 64 KB, two a CU, for grids of more tiles than CUs
// (512 experts at 128 and 512 tokens: 49.5 against 2 x 12 us per launch).
constexpr int kGemmBufs = 2;
template <int kTileK, int kTileT>
__global__ __launch_bounds__(512) void route_gemm_kernel(BatchedArgs a) {
    constexpr int kTQ = kTileT / 4;  // tokens per thread group
    static_assert((kTileE + kTileT) % 8 == 0, "every wave copies as many rows");
    __shared__ __align__(16) float wl[kGemmBufs][kTileE][kTileK];
    __shared__ __align__(16) float xl[kGemmBufs][kTileT][kTileK];
    constexpr int n = kRouteN, kSteps = n / kTileK;
    static_assert(kSteps >= kGemmBufs, "the ring is filled before the first step");
    constexpr int kRowsPerWave = (kTileE + kTileT) / 8 * (kTileK / 256);  // 1 KB copies each wave issues per step
    const int tid = threadIdx.x, q = tid >> 5, l = tid & 31, wave = wave_index(), lane = tid & 63;
    const int e0 = blockIdx.x * kTileE, t0 = blockIdx.y * kTileT;
    const int re = (q & 3) * 4, rt = (q >> 2) * kTQ;  // this group's 4 experts and kTQ tokens within the tile
    float acc[4][kTQ];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < kTQ; ++j) acc[i][j] = 0.0f;
    // 16 + TT rows of 1 KB per step: expert rows then token rows, one wave per 8 rows;
    // rows past the end repeat the last one (their results are not stored).  The
    // next steps' rows are in flight while the current one is dotted.  A shared
    // expert's gate row is not a row here: the tails kernel forms its logit,
    // which keeps 512 (256) routed experts at a whole number of rounds of tiles.
    const int er = a.E;
    auto issue = [&](int k0, int buf) {
        for (int r = wave; r < kTileE + kTileT; r += 8) {
            const int row = min(e0 + r, er - 1);
            const float *src = r < kTileE ? a.router + (size_t)row * n
                                          : a.fx + (size_t)min(t0 + r - kTileE, a.M - 1) * n;
            float *dst = r < kTileE ? wl[buf][r] : xl[buf][r - kTileE];
#pragma unroll
            for (int ck = 0; ck < kTileK / 256; ++ck)
                dma_chunk(reinterpret_cast<uint8_t *>(dst + 256 * ck), reinterpret_cast<const uint8_t *>(src + k0 + 256 * ck));
        }
    };
#pragma unroll
    for (int b = 0; b < kGemmBufs - 1; ++b) issue(b * kTileK, b);
#pragma unroll 1
    for (int st = 0; st < kSteps; ++st) {
        const int buf = st % kGemmBufs;
        const int nx = st + kGemmBufs - 1;
        if (nx < kSteps) issue(nx * kTileK, nx % kGemmBufs);
        // this step's copies landed: the wave's newer copies (up to kGemmBufs - 1 steps) may still fly
        const int newer = min(kSteps - 1 - st, kGemmBufs - 1);
        if (newer == 3)
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * kRowsPerWave) : "memory");
        else if (newer == 2)
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * kRowsPerWave) : "memory");
        else if (newer == 1)
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kRowsPerWave) : "memory");
        else
            lds_dma_wait();
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kTileK / 32; ++i) {
            float wv[4], xv[kTQ];
#pragma unroll
            for (int r = 0; r < 4; ++r) wv[r] = wl[buf][re + r][32 * i + l];
#pragma unroll
            for (int t = 0; t < kTQ; ++t) xv[t] = xl[buf][rt + t][32 * i + l];
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int t = 0; t < kTQ; ++t) acc[r][t] = fmaf(wv[r], xv[t], acc[r][t]);
        }
        __syncthreads();  // every wave is done with this buffer before it is refilled
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int t = 0; t < kTQ; ++t) {
            float v = acc[r][t];
            v = v + __shfl_xor(v, 16);  // accumulators l and l + 16
            v = row16_ggml_fold(v);
            const int e = e0 + re + r, tok = t0 + rt + t;
            if (l == 0 && e < a.E && tok < a.M) a.logits[(size_t)tok * a.E + e] = v;
        }
    (void)lane;
}

// w . x over kRouteN elements in the router's order (lane l of 32 owns
// elements l, l + 32, ...; ggml's f32 dot fold), from memory; every lane of
// the wave returns it.
__device__ __forceinline__ float router_order_dot(const float *w, const float *x) {
    const int l = threadIdx.x & 31;
    float acc = 0.0f;
#pragma unroll 16
    for (int i = 0; i < kRouteN; i += 32) acc = fmaf(w[i + l], x[i + l], acc);
    acc = acc + __shfl_xor(acc, 16);
    acc = acc + __shfl_xor(acc, 8);
    acc = acc + __shfl_xor(acc, 4);
    acc = acc + __shfl_xor(acc, 1);
    acc = acc + __shfl_xor(acc, 2);
    return acc;
}

// One token per workgroup of 640 threads: wave 0 runs the router tail
// (softmax, top-k, renorm) on the token's logits, wave b + 1 forms Q8_K of
// block b of its fx, and wave 9 the shared expert's gate logit.
// The pair's expert for the grouping: its id clamped into range (an id out of
// range counts as expert 0), or -1 where an earlier slot of the token holds the
// same clamped id, so that a token joins a group once.  ids: the token's k ids
// in lanes 0..k-1 of the calling wave.
__device__ __forceinline__ int pair_expert(int id, int j, int k, int n_ids) {
    const int e = (id < 0 || id >= n_ids) ? 0 : id;
    bool first = true;
    for (int i = 0; i < k; ++i) {
        const int o = __shfl(e, i);
        first = first && !(i < j && o == e);
    }
    return first ? e : -1;
}

// One token per workgroup of 64 (nb + 1) threads: wave 0 runs the router tail
// (softmax, top-k, renorm) on the token's logits and writes the pairs' experts
// for the grouping from the selection it holds; wave b + 1 forms Q8_K of block
// b of its fx.
__global__ __launch_bounds__(640) void route_tails_kernel(BatchedArgs a) {
    constexpr int nb = kRouteN / QK;
    static_assert(64 * (nb + 2) == 640, "a tail wave, a wave per fx block and a shared-gate wave");
    const int t = blockIdx.x, wave = wave_index(), lane = threadIdx.x & 63;
    if (wave == 0) {
        const int id = router_tail<false>(a.logits, a.E, a.k, a.renorm, a.sel, a.wsel, t);
        const int e = pair_expert(lane < a.k ? id : 0, lane, a.k, a.n_ids);
        const int kk = a.k + a.sh;  // pair (t, k): the shared expert, id n_ids
        if (lane < kk) a.pexp[(size_t)t * kk + lane] = lane < a.k ? e : a.n_ids;
    } else if (wave <= nb) {
        const int b = wave - 1;
        quantize_x(a, a.fx + (size_t)t * kRouteN + b * QK, q8(a.q8x) + (size_t)t * nb + b);
    } else if (a.sh) {
        const float v = router_order_dot(a.sh_gate_inp, a.fx + (size_t)t * kRouteN);
        if (lane == 0) a.sgl[t] = v;
    }
}

// Caller ids of a prefill-sized batch, one token per workgroup of 512 threads:
// wave b forms Q8_K of block b; wave 0 finds each slot's first occurrence of its
// id within the token (ysrc) and whether the token has an id out of range
// (bad), and writes the pairs' experts for the grouping (none for a bad token
// or a repeated id).
__global__ __launch_bounds__(512) void prep_ids_large_kernel(BatchedArgs a) {
    constexpr int nb = kRouteN / QK;
    const int t = blockIdx.x, wave = wave_index(), lane = threadIdx.x & 63, k = a.k;
    if (wave == 0) {
        const int id = lane < k ? a.sel[(size_t)t * k + lane] : 0;
        const bool bad = __any(lane < k && (id < 0 || id >= a.n_ids));
        int first = lane;
        for (int i = k - 1; i >= 0; --i) {
            const int o = __shfl(id, i);
            if (i < lane && o == id) first = i;
        }
        const int kk = k + a.sh;  // pair (t, k): the shared expert, id n_ids
        if (lane < k) {
            a.ysrc[(size_t)t * k + lane] = first;
            a.pexp[(size_t)t * kk + lane] = (bad || first != lane) ? -1 : id;
        } else if (lane < kk) {
            a.pexp[(size_t)t * kk + lane] = a.n_ids;
        }
        if (lane == 0) a.bad[t] = bad ? 1 : 0;
    }
    if (wave < nb) quantize_x(a, a.fx + (size_t)t * kRouteN + wave * QK, q8(a.q8x) + (size_t)t * nb + wave);
    if (a.sh && wave == 1) {
        const float v = router_order_dot(a.sh_gate_inp, a.fx + (size_t)t * kRouteN);
        if (lane == 0) a.sgl[t] = v;
    }
}

// The grouping of a prefill-sized batch, in one workgroup: the pairs' experts
// are copied into LDS first, so every pass reads them from there.
// The same order with every chunk's masks formed in one pass (when the
// chunks' masks of all experts fit kGroupChunkWords): chunk c (tokens
// [32 c, 32 c + 32)) of expert e has mask cm[c E + e] and starts at cb[c E + e]
// within the expert's run, so a pair's place is its expert's first place, its
// chunk's start and the tokens of its chunk before it that select the expert.
// Three barriers in all, where the chunk loop takes four per chunk.
constexpr int kGroupChunkWords = 8448;  // 16 chunks of 32 tokens x 528 experts
__device__ void group_large_chunks(const BatchedArgs &a, GroupLds &g, const int *pe, unsigned *cm, int *cb,
                                   int *sorted) {
    const int tid = threadIdx.x, nt = blockDim.x, E = a.n_ids + a.sh, k = a.k + a.sh, P = a.M * k;
    const int nch = (a.M + 31) >> 5;
    for (int e = tid; e < E; e += nt) g.cnt[e] = 0u;
    for (int i = tid; i < nch * E; i += nt) cm[i] = 0u;
    __syncthreads();
    for (int p = tid; p < P; p += nt) {
        const int e = pe[p];
        if (e < 0) continue;
        const int t = p / k;
        atomicAdd(&g.cnt[e], 1u);
        atomicOr(&cm[(t >> 5) * E + e], 1u << (t & 31));
    }
    __syncthreads();
    if (tid < 64) {
        group_units(a, g);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the records are written before their token bytes
    } else {
        for (int e = tid - 64; e < E; e += nt - 64) {
            int run = 0;
            for (int c = 0; c < nch; ++c) {
                cb[c * E + e] = run;
                run += __popc(cm[c * E + e]);
            }
        }
    }
    __syncthreads();
    for (int p = tid; p < P; p += nt) {
        const int e = pe[p];
        if (e < 0) continue;
        const int t = p / k, c = t >> 5;
        const int c0 = cb[c * E + e] + __popc(cm[c * E + e] & ((1u << (t & 31)) - 1u));  // its place in the group
        sorted[g.base[e] + c0] = t | (p - t * k) << 16;
        unit_token(a, g, e, c0, t);
    }
}

// The pairs are sorted into LDS (token | slot << 16 at each sorted place) and
// copied out in order: scattered 4-byte stores from one CU took 3 us at 4,096
// pairs, the copy a fraction of that.
__global__ __launch_bounds__(1024) void group_kernel(BatchedArgs a) {
    __shared__ GroupLds g;
    __shared__ int pe[kBatchedMaxTokensLarge * kMaxK];
    __shared__ int sorted[kBatchedMaxTokensLarge * kMaxK];
    __shared__ unsigned cm[kGroupChunkWords];
    __shared__ int cb[kGroupChunkWords];
    const int P = a.M * (a.k + a.sh);
    for (int p = threadIdx.x; p < P; p += blockDim.x) pe[p] = a.pexp[p];
    __syncthreads();
    if (((a.M + 31) >> 5) * (a.n_ids + a.sh) <= kGroupChunkWords)
        group_large_chunks(a, g, pe, cm, cb, sorted);
    else
        group_large(a, g, pe, sorted);
    __syncthreads();
    for (int i = threadIdx.x; i < g.total; i += blockDim.x) {
        const int v = sorted[i];
        a.ptok[i] = v & 0xffff;
        a.pslot[i] = v >> 16;
    }
}

// -- caller ids: Q8_K of fx (workgroups 0..M-1, a wave per block) and the
// grouping (workgroup M): each pair's first occurrence of its id within the
// token, tokens with an id out of range, then the groups as for routed ids.
// The counterpart of the verify step's mul_mat_id over the slot pool with the
// host's ids (src/run_specloop.cpp:116-139), where a token's padding repeats an
// id with weight 0.
__global__ __launch_bounds__(512) void prep_ids_kernel(BatchedArgs a) {
    constexpr int nb = kRouteN / QK;
    const int wave = wave_index();
    if ((int)blockIdx.x < a.M) {
        const int t = blockIdx.x;
        for (int b = wave; b < nb; b += 8)
            quantize_x(a, a.fx + (size_t)t * kRouteN + b * QK, q8(a.q8x) + (size_t)t * nb + b);
        if (a.sh && wave == 0) {
            const float v = router_order_dot(a.sh_gate_inp, a.fx + (size_t)t * kRouteN);
            if ((threadIdx.x & 63) == 0) a.sgl[t] = v;
        }
        return;
    }
    __shared__ int bad_s[kMaxTok];
    __shared__ int ysrc_s[kMaxTok * kMaxK];
    __shared__ int sel_s[kMaxTok * kMaxK];
    __shared__ GroupLds g;
    const int tid = threadIdx.x, P = a.M * a.k;
    for (int t = tid; t < a.M; t += blockDim.x) bad_s[t] = 0;
    for (int p = tid; p < P; p += blockDim.x) sel_s[p] = a.sel[p];
    __syncthreads();
    for (int p = tid; p < P; p += blockDim.x) {
        const int t = p / a.k, j = p % a.k;
        const int e = sel_s[p];
        if (e < 0 || e >= a.n_ids) bad_s[t] = 1;
        int first = j;
        for (int i = j - 1; i >= 0; --i)
            if (sel_s[t * a.k + i] == e) first = i;
        ysrc_s[p] = first;
        a.ysrc[p] = first;  // for the combine launch
    }
    __syncthreads();
    for (int t = tid; t < a.M; t += blockDim.x) a.bad[t] = bad_s[t];
    group_by_expert(a, g, sel_s, ysrc_s, bad_s);
}

// -- combine: out[t][d] = (sum_j w[t][j] * y[t][j][d]) + res[t][d], j ascending --
__global__ __launch_bounds__(256) void combine_kernel(BatchedArgs a) {
    const int t = blockIdx.y;
    const int d = blockIdx.x * blockDim.x + threadIdx.x;
    if (d >= a.n_embd) return;
    if (a.bad && a.bad[t]) {  // an id outside the pool or expert set: the token's row is poisoned
        a.out[(size_t)t * a.n_embd + d] = __builtin_nanf("");
        return;
    }
    const int kk = a.k + a.sh;
    // every load is issued before the first is used: one memory latency, not k
    float w[kMaxK], y[kMaxK];
#pragma unroll
    for (int j = 0; j < kMaxK; ++j) {
        if (j < a.k) {
            const int js = a.ysrc ? a.ysrc[t * a.k + j] : j;  // a repeated id takes its first output
            w[j] = a.wsel[t * a.k + j];
            y[j] = a.ybuf[((size_t)t * kk + js) * a.n_embd + d];
        }
    }
    const float ysh = a.sh ? a.ybuf[((size_t)t * kk + a.k) * a.n_embd + d] : 0.0f;
    const float r = a.res[(size_t)t * a.n_embd + d];
    float acc = 0.0f;
#pragma unroll
    for (int j = 0; j < kMaxK; ++j)
        if (j < a.k) acc = acc + w[j] * y[j];
    if (a.sh) {  // + sigmoid(gate logit) * shared expert output
        const float sg = 1.0f / (1.0f + expf(-a.sgl[t]));
        acc = acc + ysh * sg;
    }
    a.out[(size_t)t * a.n_embd + d] = acc + r;
}

// The same for prefill-sized batches.
__global__ __launch_bounds__(256) void pf_combine_kernel(BatchedArgs a) {
    // four consecutive elements a thread (n_embd is a multiple of 1024): at
    // hundreds of tokens the wider loads pay; at 16 tokens the one-element
    // form of the batched path keeps more workgroups in flight
    const int t = blockIdx.y;
    const int d = 4 * (blockIdx.x * blockDim.x + threadIdx.x);
    if (d >= a.n_embd) return;
    float4 *o = reinterpret_cast<float4 *>(a.out + (size_t)t * a.n_embd + d);
    if (a.bad && a.bad[t]) {  // an id outside the pool or expert set: the token's row is poisoned
        const float nan = __builtin_nanf("");
        *o = make_float4(nan, nan, nan, nan);
        return;
    }
    const int kk = a.k + a.sh;
    // every load is issued before the first is used: one memory latency, not k
    float w[kMaxK];
    float4 y[kMaxK];
#pragma unroll
    for (int j = 0; j < kMaxK; ++j) {
        if (j < a.k) {
            const int js = a.ysrc ? a.ysrc[t * a.k + j] : j;  // a repeated id takes its first output
            w[j] = a.wsel[t * a.k + j];
            y[j] = *reinterpret_cast<const float4 *>(a.ybuf + ((size_t)t * kk + js) * a.n_embd + d);
        }
    }
    const float4 ysh = a.sh ? *reinterpret_cast<const float4 *>(a.ybuf + ((size_t)t * kk + a.k) * a.n_embd + d)
                            : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const float4 r = *reinterpret_cast<const float4 *>(a.res + (size_t)t * a.n_embd + d);
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int j = 0; j < kMaxK; ++j) {
        if (j < a.k) {
            acc.x = acc.x + w[j] * y[j].x;
            acc.y = acc.y + w[j] * y[j].y;
            acc.z = acc.z + w[j] * y[j].z;
            acc.w = acc.w + w[j] * y[j].w;
        }
    }
    if (a.sh) {  // + sigmoid(gate logit) * shared expert output
        const float sg = 1.0f / (1.0f + expf(-a.sgl[t]));
        acc.x = acc.x + ysh.x * sg;
        acc.y = acc.y + ysh.y * sg;
        acc.z = acc.z + ysh.z * sg;
        acc.w = acc.w + ysh.w * sg;
    }
    *o = make_float4(acc.x + r.x, acc.y + r.y, acc.z + r.z, acc.w + r.w);
}

}  // namespace

bool batched_shape_compiled(int gu_type, int n_embd, int d_type, int n_ff) {
    return (gu_type == kTypeQ4K || gu_type == kTypeQ3K) && n_embd == 2048 &&
           (n_ff == 768 || n_ff == 1024 || n_ff == 512) &&
           (d_type == kTypeQ4K || d_type == kTypeQ6K || (d_type == kTypeQ5K && n_ff != 768));
}

namespace {

hipError_t launch_combine(const BatchedArgs &a, hipStream_t s) {
    if (a.M > kMaxTok)
        hipLaunchKernelGGL(pf_combine_kernel, dim3((a.n_embd + 1023) / 1024, a.M), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL(combine_kernel, dim3((a.n_embd + 255) / 256, a.M), dim3(256), 0, s, a);
    return hipGetLastError();
}

// The launches after the grouping.
hipError_t launch_groups(const BatchedArgs &a, hipStream_t s) {
    if (hipError_t e = launch_expert_units(a, s); e != hipSuccess) return e;
    return launch_combine(a, s);
}

bool args_ok(const BatchedArgs &a) {
    return a.M >= 1 && a.M <= kBatchedMaxTokensLarge && a.n_embd == kRouteN &&
           (a.gu_type == kTypeQ4K || a.gu_type == kTypeQ3K) &&
           a.k + a.sh <= kMaxK && a.n_ids >= 1 && a.n_ids + a.sh <= kMaxExperts && a.E + a.sh <= kMaxExperts &&
           (!a.sh || (a.sh == 1 && a.sh_gate && a.sh_up && a.sh_down && a.sh_gate_inp && a.sgl)) &&
           a.ptok && a.pslot && a.pexp && a.units;
}

}  // namespace

// How the batch's groups are cut into units (unit_shift).  Figures: us/layer of
// ffn_combine_batched with uniform ids and, after the bar, every token on the same
// experts; P pairs over n experts.
//
// Dots for the small groups while experts hold up to two pairs on average: a dot
// costs less than folding a row's weights for 16 MFMA columns.  In the down
// launch, which then forms Q8_K(h) itself, only for the verify-sized batches: its
// dots and the forming grow with the pairs, a launch for Q8_K(h) hardly does.
// Dots in both launches / in gate/up alone / nowhere:
//   Q3_K / Q5_K, 64 experts:    M = 8 52 / 61 / 65, M = 16 (2 n) 80 / 87 / 82, M = 24 102 / 107 / 88
//   Q4_K, 64:                   M = 8 43 / 48 / 50, M = 16 (2 n) 60 / 62 / 62, M = 24 75 / 74 / 66
//   Q4_K / Q6_K, 128:           M = 16 65 / 68 / 76, M = 32 (2 n) 90 / 91 / 94 | 38 / 30 / 29, M = 40 102 / 103 / 100
//   Q4_K / Q5_K, 256, a shared: M = 32 77 / 80 / 89 | 39 / 32 / 30, M = 64 (2 n) 115 / 113 / 116 | 54 / 41 / 38
//   Q4_K / Q6_K, 512, a shared: M = 32 105 / 102 / 118 | 42 / 33 / 32, M = 40 125 / 118 / 142 | 54 / 40 / 38,
//                               M = 102 (2 n) 216 / 206 / 216 | 89 / 52 / 49
// A group of kMfmaPairs = 8 pairs goes to MFMA all the same (tokens of one prompt
// or draft share experts).  Lines of 6 / 8 / 10 / 12, tokens that pick among
// 2 k experts: 128 experts M = 8 35.9 / 33.5 / 33.3 / 33.5, M = 16 38.6 / 41.4 /
// 43.0 / 43.7; 512 M = 24 40.1 / 40.1 / 43.2 / 46.1; Q3_K M = 16 52 / 50 / 61 / 70.
//
// Units of 16 and 32 by group until experts hold 21 pairs on average, then of
// 64: small ones keep more weights in flight, large ones read and fold an
// expert's weights once for more pairs.  16 and 32 / 64:
//   256 experts, M = 128 (4 n):  137 / 161 | 48 / 52
//   512, M = 512 (10 n):         296 / 306 | 129 / 117
//   64, M = 128 (16 n):          92 / 97 | 54 / 52
//   128, M = 256 (16 n):         133 / 135 | 73 / 65
//   64, M = 256 (32 n):          127 / 118 | 88 / 82
static int units_mode(const BatchedArgs &a) {
    const int P = a.M * a.k, n = a.n_ids;
    if (a.M <= kMaxDotTokens && P <= 2 * n) return a.M <= kMaxTok ? kUnitsDots : kUnitsDotGateUp;
    return P <= 21 * n ? kUnitsMixed : kUnitsLarge;
}
static BatchedArgs with_units(const BatchedArgs &a) {
    BatchedArgs r = a;
    r.units_mode = units_mode(a);
    const int least = r.units_mode <= kUnitsDotGateUp ? kDotTokens : r.units_mode == kUnitsMixed ? kUnitTokensMin : kUnitTokens;
    r.max_units = prefill_max_units(a.M, a.k + a.sh, a.n_ids + a.sh, least);
    return r;
}

// Batches of up to 32 tokens route, group and form Q8_K(fx) in one launch;
// larger ones in three, the router as a matrix product.  Both then run units of
// sorted pairs (prefill.hip).
hipError_t launch_batched(const BatchedArgs &args, hipStream_t s) {
    const BatchedArgs a = with_units(args);
    if (!args_ok(a) || a.ysrc || a.n_ids != a.E || (a.M + kRouteTok - 1) / kRouteTok > kBatchedCounters - 1)
        return hipErrorInvalidValue;
    if (a.M > kMaxTok) {
        const unsigned et = (a.E + kTileE - 1) / kTileE;
        const dim3 rg(et, (a.M + 15) / 16);
        if (rg.x * rg.y > 256)  // more tiles than CUs: two workgroups a CU
            hipLaunchKernelGGL((route_gemm_kernel<256, 16>), rg, dim3(512), 0, s, a);
        else if (rg.x * rg.y > 128)
            hipLaunchKernelGGL((route_gemm_kernel<512, 16>), rg, dim3(512), 0, s, a);
        else  // at most half the CUs with 16-token tiles: 8-token ones, at most one a CU
            hipLaunchKernelGGL((route_gemm_kernel<512, 8>), dim3(et, (a.M + 7) / 8), dim3(512), 0, s, a);
        hipLaunchKernelGGL(route_tails_kernel, dim3(a.M), dim3(640), 0, s, a);
        hipLaunchKernelGGL(group_kernel, dim3(1), dim3(1024), 0, s, a);
        return launch_groups(a, s);
    }
    // row workgroups: a remainder of one row joins the last workgroup
    const int nr = a.E + a.sh, ntg = (a.M + kRouteTok - 1) / kRouteTok;
    auto row_groups = [nr](int R) { return nr > R && nr % R == 1 ? nr / R : (nr + R - 1) / R; };
    if (a.M > 8)
        hipLaunchKernelGGL(route_kernel<4>, dim3(row_groups(4), ntg), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL(route_kernel<2>, dim3(row_groups(2), ntg), dim3(256), 0, s, a);
    return launch_groups(a, s);
}

hipError_t launch_batched_ids(const BatchedArgs &args, hipStream_t s) {
    const BatchedArgs a = with_units(args);
    if (!args_ok(a) || !a.ysrc || !a.bad) return hipErrorInvalidValue;
    if (a.M > kMaxTok) {
        hipLaunchKernelGGL(prep_ids_large_kernel, dim3(a.M), dim3(512), 0, s, a);
        hipLaunchKernelGGL(group_kernel, dim3(1), dim3(1024), 0, s, a);
        return launch_groups(a, s);
    }
    hipLaunchKernelGGL(prep_ids_kernel, dim3((unsigned)a.M + 1), dim3(512), 0, s, a);
    return launch_groups(a, s);
}

}  // namespace hoard
