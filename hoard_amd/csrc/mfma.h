// Pieces shared by the int8 MFMA kernels: packed K-quant scales, bytes of
// words, reads of 2-byte aligned LDS blocks.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "qblocks.h"
#include "rowdot.h"

namespace hoard {

typedef int v4i __attribute__((ext_vector_type(4)));

// The 6-bit scales (sc) and mins (mn) of a Q4_K header, four per word: byte
// s of sc[0] / mn[0] belongs to sub-block s, byte s of sc[1] / mn[1] to s + 4.
__device__ __forceinline__ void q4k_scales_packed(const uint4 &hd, uint32_t sc[2], uint32_t mn[2]) {
    sc[0] = hd.y & 0x3f3f3f3fu;
    mn[0] = hd.z & 0x3f3f3f3fu;
    sc[1] = (hd.w & 0x0f0f0f0fu) | ((hd.y >> 2) & 0x30303030u);
    mn[1] = ((hd.w >> 4) & 0x0f0f0f0fu) | ((hd.z >> 2) & 0x30303030u);
}

__device__ __forceinline__ int byte_of(uint32_t w, int i) { return (int)((w >> (8 * i)) & 0xffu); }

// 8 bytes at a 2-byte aligned LDS address.
__device__ __forceinline__ uint2 lds_u64_a2(const uint8_t *p) {
    // aligned base by pointer arithmetic, so that the compiler still sees an
    // LDS pointer and emits ds_read rather than flat loads
    const uint32_t sh = (uint32_t)(reinterpret_cast<uintptr_t>(p) & 3u);
    const uint32_t *w = reinterpret_cast<const uint32_t *>(p - sh);
    const uint32_t w0 = w[0], w1 = w[1], w2 = w[2];
    return make_uint2(__builtin_amdgcn_alignbyte(w1, w0, sh), __builtin_amdgcn_alignbyte(w2, w1, sh));
}

}  // namespace hoard
