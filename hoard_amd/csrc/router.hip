// Fused router tail (kernel family 1): f32 router GEMV, softmax over all
// experts, top-k, gather and optional renorm, in one launch, any shape the
// stage takes (layer.hip has the one compiled for the 2048-wide hidden).
//
// Replaces ggml_mul_mat(ffn_gate_inp, fx) + ggml_soft_max + ggml_top_k +
// ggml_get_rows (src/run_moe_stream.cpp:353-356, src/run_qwen35.cpp:556-559)
// and the host renorm (src/run_moe_stream.cpp:371-373).
//
// A launch is latency: the rows' copies, a chain of n / 32 FMAs a lane, the
// hand-off to the tail.  Four rows per workgroup go to LDS a wave each with
// their copies in flight together, kChunk elements of a row at a time; the
// dot's 32 lanes own elements l, l + 32, ... and keep one fused multiply-add
// chain each, the same 32 accumulators ggml's x86 f32 dot keeps (4 vectors x
// 8 lanes), folded in that dot's order (16, 8, 4 lanes apart, then pairs), so
// the logits are the CPU path's bit for bit.  The logits are stored and read
// at device scope (past the per-XCD L2) and a workgroup counts itself done
// once its stores are acknowledged, so no cache-flushing fence is needed; the
// last one runs softmax / top-k on one wave.  64 experts of 4096: 8.9 us a
// launch, 12.7 with one wave per two rows and fences.
#include "kernels.h"
#include "lds_dma.h"
#include "rowstream.h"
#include "router_tail.h"

namespace hoard {

namespace {

constexpr int kRows = 4;      // router rows per workgroup, a wave each
constexpr int kChunk = 4096;  // elements of a row in LDS at a time (80 KB with x: two workgroups a CU)

__global__ __launch_bounds__(64 * kRows) void router_kernel(RouterArgs a) {
    __shared__ __align__(16) float xl[kChunk];
    __shared__ __align__(16) float wl[kRows][kChunk];
    __shared__ double red[kRows];
    __shared__ int last;
    const int n = a.n, E = a.E;
    const int wave = wave_index(), lane = threadIdx.x & 63, l = lane & 31;
    const int row = blockIdx.x * kRows + wave;
    const bool has = row < E;
    const float *wr = a.w + (size_t)(has ? row : 0) * n;

    float acc = 0.0f, scale = 1.0f;
    for (int c0 = 0; c0 < n; c0 += kChunk) {
        const int len = min(kChunk, n - c0);
        if (c0 > 0) __syncthreads();  // the previous chunk is dotted
        if (has)
            dma_wave_copy(reinterpret_cast<uint8_t *>(wl[wave]), reinterpret_cast<const uint8_t *>(wr + c0),
                          len * (int)sizeof(float));
        for (int i = 4 * threadIdx.x; i < len; i += 4 * 64 * kRows)
            *reinterpret_cast<u32x4 *>(xl + i) = *reinterpret_cast<const u32x4_a4 *>(a.xin + c0 + i);
        if (c0 == 0 && a.xin_is_residual) {
            // rms_norm: mean of x*x accumulated in double, scale = 1/sqrtf(mean + eps)
            double ss = 0.0;
            for (int i = threadIdx.x; i < n; i += 64 * kRows) {
                const float v = a.xin[i];
                ss += (double)(v * v);
            }
            ss = wave_sum_d(ss);
            if (lane == 0) red[wave] = ss;
            __syncthreads();
            const float mean = (float)(((red[0] + red[1]) + (red[2] + red[3])) / (double)n);
            scale = 1.0f / sqrtf(mean + a.eps);
            if (blockIdx.x == 0)
                for (int i = threadIdx.x; i < n; i += 64 * kRows) a.fx_out[i] = a.xin[i] * scale;
        }
        lds_dma_wait();
        __syncthreads();
        if (has && lane < 32) {
            const float *wp = wl[wave] + l, *xp = xl + l;
#pragma unroll 16
            for (int i = 0; i < len; i += 32) acc = fmaf(wp[i], xp[i] * scale, acc);
        }
    }
    if (has && lane < 32) {
        acc = acc + __shfl_xor(acc, 16);
        acc = row16_ggml_fold(acc);
        if (l == 0) __hip_atomic_store(a.logits + row, acc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the logits are acknowledged

    // ---- the last workgroup runs the tail ----
    __syncthreads();
    if (threadIdx.x == 0)
        last = __hip_atomic_fetch_add(&a.counters[0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
    __syncthreads();
    if (!last) return;
    if (wave == 0) {
        const int id = router_tail<true>(a.logits, E, a.k, a.renorm, a.sel, a.wsel, 0);
        if (a.sel_host && lane < a.k) a.sel_host[lane] = id;
    }
    if (threadIdx.x == 0) __hip_atomic_store(&a.counters[0], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace

hipError_t launch_router(const RouterArgs &a, hipStream_t s) {
    if (a.M != 1) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL(router_kernel, dim3((unsigned)((a.E + kRows - 1) / kRows)), dim3(64 * kRows), 0, s, a);
    return hipGetLastError();
}

}  // namespace hoard
