// The slot pool's upload step of an on-demand layer (src/run_moe_stream.cpp:379-420):
// the missed experts' records come over PCIe by a kernel on the compute
// stream instead of copies on streams of their own.
//
// The link bounds it either way (8 records of 3.06 MB: 442 us by a kernel of
// 16 to 64 workgroups, 55.4 GB/s; 436 by hipMemcpyAsync on three streams); what
// the kernel saves is what stands around the copies: the event waits between
// the streams, the copies' start-up, and the copy of the slot ids, which
// travel in the kernel's arguments.  Few workgroups: the link needs about 256 KB
// in flight, and more of them only contend (32 a record: 465 us).
#include "kernels.h"

namespace hoard {

namespace {

constexpr int kThreads = 256;
constexpr int kAhead = 4;  // 16-byte loads a thread has in flight

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(kThreads) void slot_fill_kernel(SlotFill a, int per_record) {
    if (blockIdx.x == 0 && (int)threadIdx.x < a.n_ids) a.slot_dev[threadIdx.x] = a.slot[threadIdx.x];
    const int r = blockIdx.x / per_record, w = blockIdx.x - r * per_record;
    if (r >= a.n) return;  // no record: the ids alone
    const u32x4 *src = reinterpret_cast<const u32x4 *>(a.src[r]);
    u32x4 *dst = reinterpret_cast<u32x4 *>(a.dst[r]);
    const size_t n = a.bytes / 16, step = (size_t)per_record * kThreads * kAhead;
    for (size_t i = (size_t)w * kThreads * kAhead + threadIdx.x; i < n; i += step) {
        u32x4 v[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
            if (i + kThreads * u < n) v[u] = __builtin_nontemporal_load(src + i + kThreads * u);
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
            if (i + kThreads * u < n) dst[i + kThreads * u] = v[u];
    }
}

}  // namespace

hipError_t launch_slot_fill(const SlotFill &a, hipStream_t s) {
    if (a.n < 0 || a.n > kMaxSlotIds || a.n_ids < 0 || a.n_ids > kMaxSlotIds || a.bytes % 16) return hipErrorInvalidValue;
    // 16 workgroups in all, or four a record: one record 65 us with 16, 86 with four
    const int per_record = a.n >= 4 ? 4 : a.n > 0 ? 16 / a.n : 1;
    const int grid = a.n > 0 ? a.n * per_record : 1;
    hipLaunchKernelGGL(slot_fill_kernel, dim3((unsigned)grid), dim3(kThreads), 0, s, a, per_record);
    return hipGetLastError();
}

}  // namespace hoard
