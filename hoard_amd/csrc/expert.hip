// Grouped dequant-GEMV over the selected experts (kernel family 2) and the
// fused weighted combine (family 4), one token, any shape the stage takes.
//
// Replaces graph B of src/run_moe_stream.cpp:431-438 (per expert:
// mul_mat(gate), mul_mat(up), mul(silu(g), u), mul_mat(down), concat) plus the
// shared expert of src/run_qwen35.cpp:658-666, and the host combine at
// src/run_moe_stream.cpp:447 / src/run_qwen35.cpp:675-676.
//
// Both kernels are bound by the weight stream.  A wave streams 8 rows from
// memory into registers (rowstream.h), the first blocks' loads issued before
// the activation's Q8_K blocks are formed in LDS, so the formation and the
// barrier behind it pass while they fly.  Against copying whole tiles through
// registers into LDS first (a few loads in flight per CU): 8 of 64 experts of
// 4096 x 1536 (Q4_K, Q6_K down), gate/up 33.5 -> 15.6 us a launch (56.6 MB,
// 3.6 TB/s), down 65.2 -> 15.4 us (41.3 MB, 2.7 TB/s).
#include "kernels.h"
#include "lds_dma.h"
#include "qblocks.h"
#include "router_tail.h"
#include "rowstream.h"
#include "wave.h"

namespace hoard {

namespace {

constexpr int kWaveRows = 8;   // rows a wave streams, one 8-lane group each
constexpr size_t kMaxLds = 163840 - 2048;  // dynamic LDS of a workgroup, beside the static words

__device__ __forceinline__ size_t row_bytes(int type, int cols) {
    return (size_t)(cols / QK) * (size_t)kquant_block_bytes(type);
}

// The dot of the lane group's row (row grp of the 8 at base) with q; prep()
// runs once the rows' first loads are issued.
template <int T, class P>
__device__ __forceinline__ float stream_row_t(const uint8_t *base, const Q8L *q, int nb, P prep) {
    const int lane = threadIdx.x & 63, t = lane & 7;
    const uint32_t off = (uint32_t)(lane >> 3) * (uint32_t)(nb * QType<T>::bytes);
    RowStream<T> rs;
    rs.begin(base, off, nb, t);
    prep();
    return rs.finish(base, off, q, nb, t);
}
// T: the type of every matrix the kernel meets, or 0 where they differ (type
// is the same in every lane of the wave).
template <int T, class P>
__device__ __forceinline__ float stream_row(int type, const uint8_t *base, const Q8L *q, int nb, P prep) {
    if constexpr (T != 0) {
        return stream_row_t<T>(base, q, nb, prep);
    } else {
        switch (type) {
        case kTypeQ4K: return stream_row_t<kTypeQ4K>(base, q, nb, prep);
        case kTypeQ5K: return stream_row_t<kTypeQ5K>(base, q, nb, prep);
        case kTypeQ3K: return stream_row_t<kTypeQ3K>(base, q, nb, prep);
        default: return stream_row_t<kTypeQ6K>(base, q, nb, prep);
        }
    }
}

// The selection of a small router, by every workgroup that needs it: all rows
// and x go to LDS with their copies in flight together, a half-wave forms each
// row in the router's order (router.hip) and one wave runs the tail.
__device__ void route_in_place(const GateUpArgs &a, float *lds, int32_t *sel, float *w) {
    const int wave = wave_index(), lane = threadIdx.x & 63, l = lane & 31, nw = (int)(blockDim.x >> 6);
    const int n = a.n_embd;
    float *xl = lds, *wl = lds + n, *lg = wl + (size_t)a.E * n;
    for (int e = wave; e < a.E; e += nw)
        dma_wave_copy(reinterpret_cast<uint8_t *>(wl + (size_t)e * n), reinterpret_cast<const uint8_t *>(a.router + (size_t)e * n),
                      n * (int)sizeof(float));
    for (int i = 4 * threadIdx.x; i < n; i += 4 * blockDim.x)
        *reinterpret_cast<u32x4 *>(xl + i) = *reinterpret_cast<const u32x4_a4 *>(a.fx + i);
    lds_dma_wait();
    __syncthreads();
    for (int e0 = 2 * wave; e0 < a.E; e0 += 2 * nw) {
        const int e = e0 + (lane >> 5);
        const float *wp = wl + (size_t)(e < a.E ? e : e0) * n + l, *xp = xl + l;
        float acc = 0.0f;
#pragma unroll 16
        for (int i = 0; i < n; i += 32) acc = fmaf(wp[i], xp[i], acc);
        acc = acc + __shfl_xor(acc, 16);
        acc = row16_ggml_fold(acc);
        if (l == 0 && e < a.E) lg[e] = acc;
    }
    __syncthreads();
    if (wave == 0) router_tail<false>(lg, a.E, a.k, a.renorm, sel, w, 0);
    __syncthreads();
}

// ---------------------------------------------------------------------------
// gate/up + SwiGLU.  grid = (rows_max / R, k + has_shared, plus a workgroup row
// for the shared expert's gate); block = 64 * R / 4: R / 8 waves stream the
// gate rows and R / 8 the up rows.
// ---------------------------------------------------------------------------
template <int T, bool ROUTE>
__global__ __launch_bounds__(512) void gateup_kernel(GateUpArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ float gu[64];
    __shared__ int32_t sel_s[16];
    __shared__ float w_s[16];
    const int wave = wave_index(), lane = threadIdx.x & 63, t = lane & 7, grp = lane >> 3;
    const int nw = (int)(blockDim.x >> 6), R = nw / 2 * kWaveRows;
    const int j = blockIdx.y;
    const bool shared = j >= a.k;
    if (j > a.k) {
        // sigmoid gate of the shared expert: f32 dot in the router's lane order
        if (blockIdx.x == 0 && threadIdx.x < 32) {
            float acc = 0.0f;
#pragma unroll 32
            for (int i = 0; i < a.n_embd; i += 32) acc = fmaf(a.sh_gate_inp[i + lane], a.fx[i + lane], acc);
            acc = acc + __shfl_xor(acc, 16);
            acc = row16_ggml_fold(acc);
            if (lane == 0) a.sgate[0] = 1.0f / (1.0f + expf(-acc));
        }
        return;
    }
    const bool up = wave >= nw / 2;
    const MatDesc &W = shared ? (up ? a.sh_up : a.sh_gate) : (up ? a.up : a.gate);
    const int r0 = blockIdx.x * R;
    if (r0 >= W.rows) return;
    const int nb = a.n_embd / QK;
    float *hout = a.h + (size_t)j * a.hstride + r0;
    const uint8_t *src = W.base;
    if (ROUTE && !shared) {
        route_in_place(a, reinterpret_cast<float *>(smem + (size_t)nb * sizeof(Q8L)), sel_s, w_s);
        if (blockIdx.x == 0 && j == 0 && threadIdx.x < a.k) {
            a.sel[threadIdx.x] = sel_s[threadIdx.x];
            a.wsel[threadIdx.x] = w_s[threadIdx.x];
        }
    }
    if (!shared) {
        const int id = ROUTE ? __builtin_amdgcn_readfirstlane(sel_s[j]) : a.ids[j];
        if (id < 0 || id >= W.n_ids) {  // invalid id: poison this expert's rows
            if (threadIdx.x < R) hout[threadIdx.x] = __builtin_nanf("");
            return;
        }
        src += (size_t)id * W.stride;
    }
    Q8L *q8 = reinterpret_cast<Q8L *>(smem);
    WaveQuant<4> xq;
    xq.load(a.fx, wave, nb, nw);
    const int w0 = (up ? wave - nw / 2 : wave) * kWaveRows;  // the wave's first row of the R
    const float v = stream_row<T>(W.type, src + (size_t)(r0 + w0) * row_bytes(T ? T : W.type, a.n_embd), q8, nb, [&]() {
        xq.form(a.fx, q8, wave, nb, nw);
        lds_barrier();
    });
    if (t == 0) gu[(up ? R : 0) + w0 + grp] = v;
    lds_barrier();
    if (threadIdx.x < R) {
        const float g = gu[threadIdx.x], u = gu[R + threadIdx.x];
        hout[threadIdx.x] = g / (1.0f + expf(-g)) * u;
    }
}

// ---------------------------------------------------------------------------
// down + combine.  grid = n_embd / (8 G) workgroups of G waves a unit (the k
// experts, then the shared one; several units a wave where they are more than
// 16 waves): wave u G + s streams rows [8 s, 8 s + 8) of unit u.
// ---------------------------------------------------------------------------
template <int T>
__global__ __launch_bounds__(1024) void down_combine_kernel(DownArgs a, int G) {
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ float ys[17 * 4 * kWaveRows];
    __shared__ int bad;
    const int wave = wave_index(), lane = threadIdx.x & 63, t = lane & 7, grp = lane >> 3;
    const int nw = (int)(blockDim.x >> 6), R = kWaveRows * G;
    const int d0 = blockIdx.x * R;
    const int k = a.k;
    const bool has_sh = a.sh_down.base != nullptr;
    const int nu = k + (has_sh ? 1 : 0);
    const int nbh = a.down.cols / QK;
    Q8L *q8h = reinterpret_cast<Q8L *>(smem);  // unit u's blocks at u * nbh
    if (threadIdx.x == 0) bad = 0;
    lds_barrier();
    for (int w = wave; w < nu * G; w += nw) {
        const int u = w / G, s = w - u * G;
        const MatDesc &W = u < k ? a.down : a.sh_down;
        const int nb = W.cols / QK;
        const float *h = a.h + (size_t)u * a.hstride;
        const int id = u < k ? a.ids[u] : 0;
        const bool ok = u >= k || (id >= 0 && id < W.n_ids);
        if (!ok) bad = 1;
        Q8L *q = q8h + (size_t)u * nbh;
        WaveQuant<T == 0 ? 2 : 8> hq;
        hq.load(h, s, nb, G);
        const uint8_t *rows = W.base + (size_t)(ok ? id : 0) * W.stride +
                              (size_t)(d0 + kWaveRows * s) * row_bytes(T ? T : W.type, W.cols);
        const float y = stream_row<T>(W.type, rows, q, nb, [&]() {
            hq.form(h, q, s, nb, G);
            // one wave a unit: its blocks are its own; several: they form them together
            if (G > 1)
                lds_barrier();
            else
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        });
        if (t == 0) ys[u * R + kWaveRows * s + grp] = y;
    }
    lds_barrier();
    if (threadIdx.x < R) {
        const int r = threadIdx.x, d = d0 + r;
        float acc = 0.0f;
        for (int j = 0; j < k; ++j) acc = acc + a.w[j] * ys[j * R + r];
        float o = has_sh ? (acc + ys[k * R + r] * a.sgate[0]) + a.res[d] : acc + a.res[d];
        a.out[d] = bad ? __builtin_nanf("") : o;
    }
}

}  // namespace

size_t block_bytes(int type) { return (size_t)kquant_block_bytes(type); }

namespace {

size_t route_lds(const GateUpArgs &a) { return ((size_t)(a.E + 1) * a.n_embd + a.E) * sizeof(float); }

template <bool ROUTE>
hipError_t launch_gateup_t(const GateUpArgs &a, hipStream_t s) {
    const size_t lds = (size_t)(a.n_embd / QK) * sizeof(Q8L) + (ROUTE ? route_lds(a) : 0);
    if (lds > kMaxLds) return hipErrorInvalidConfiguration;
    const bool sh = a.sh_gate.base != nullptr;
    const int rows = sh && a.sh_gate.rows > a.gate.rows ? a.sh_gate.rows : a.gate.rows;
    const int units = a.k + (sh ? 1 : 0);
    // eight waves share one formation of Q8_K(fx) where that still gives every
    // CU a workgroup; fewer rows take four, for twice the workgroups
    const int waves = rows * units >= 8192 ? 8 : 4;
    const dim3 grid((unsigned)(rows / (4 * waves)), (unsigned)(units + (sh ? 1 : 0)));
    const int T = a.gate.type;
    const bool one = a.up.type == T && (!sh || (a.sh_gate.type == T && a.sh_up.type == T));
    auto *fn = !one             ? gateup_kernel<0, ROUTE>
               : T == kTypeQ4K ? gateup_kernel<kTypeQ4K, ROUTE>
               : T == kTypeQ5K ? gateup_kernel<kTypeQ5K, ROUTE>
               : T == kTypeQ3K ? gateup_kernel<kTypeQ3K, ROUTE>
                               : gateup_kernel<kTypeQ6K, ROUTE>;
    hipLaunchKernelGGL(fn, grid, dim3(64 * waves), lds, s, a);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_gateup(const GateUpArgs &a, hipStream_t s) { return launch_gateup_t<false>(a, s); }

// A router (16-byte aligned, for the LDS copies) whose rows fit LDS beside the workgroup's own blocks, in a launch of
// at most one workgroup a CU: every workgroup reads the whole router (from its
// XCD's L2 after the first), which costs less than the router's own launch and
// the boundary after it until the rows are many.  A layer, us, with the launch
// and without: n_embd 1024, 8 experts, top 2, n_ff 512 15.3 and 12.9; 2048, 6,
// 4, 1024 19.4 and 17.6; 2304, 4, 2, 2048 23.7 and 20.8; 256, 32, 16, 256 16.7
// and 15.8.  Past the lines: 256, 50, 4, 256 13.4 and 14.0 (few columns a row
// and many rows a wave); 1024, 14, 8, 2048 23.2 and 23.5; 3072, 4, 2 and a
// shared expert, 1536 23.8 and 24.0.
bool gateup_routed_ok(const GateUpArgs &a) {
    const bool sh = a.sh_gate.base != nullptr;
    const int rows = sh && a.sh_gate.rows > a.gate.rows ? a.sh_gate.rows : a.gate.rows;
    return a.router && ((uintptr_t)a.router & 15) == 0 && a.E <= 32 && rows * (a.k + sh) <= 4096 &&
           (size_t)(a.n_embd / QK) * sizeof(Q8L) + route_lds(a) <= 61440;
}
hipError_t launch_gateup_routed(const GateUpArgs &a, hipStream_t s) {
    if (!gateup_routed_ok(a)) return hipErrorInvalidConfiguration;
    return launch_gateup_t<true>(a, s);
}

hipError_t launch_down_combine(const DownArgs &a, hipStream_t s) {
    const bool has_sh = a.sh_down.base != nullptr;
    const int nu = a.k + (has_sh ? 1 : 0), nbh = a.down.cols / QK, nbs = has_sh ? a.sh_down.cols / QK : 0;
    const size_t lds = (size_t)(a.k * nbh + nbs) * sizeof(Q8L);
    if (lds > kMaxLds) return hipErrorInvalidConfiguration;
    // several waves a unit (up to 16 in all) share the formation of its Q8_K(h),
    // as long as every CU has a workgroup: 15.5 against 16.1 us at 4096 rows of
    // 8 units with two
    int G = 1;
    while (G < 4 && 2 * G * nu <= 16 && a.n_embd / (kWaveRows * 2 * G) >= 256) G *= 2;
    const int waves = nu * G < 16 ? nu * G : 16;
    const int T = a.down.type;
    auto *fn = has_sh && a.sh_down.type != T ? down_combine_kernel<0>
               : T == kTypeQ4K               ? down_combine_kernel<kTypeQ4K>
               : T == kTypeQ5K               ? down_combine_kernel<kTypeQ5K>
               : T == kTypeQ3K               ? down_combine_kernel<kTypeQ3K>
                                             : down_combine_kernel<kTypeQ6K>;
    hipLaunchKernelGGL(fn, dim3((unsigned)(a.n_embd / (kWaveRows * G))), dim3(64 * waves), lds, s, a, G);
    return hipGetLastError();
}

}  // namespace hoard
