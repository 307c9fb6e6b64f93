// Raw buffers and 16-byte LDS-DMA loads, as apply_mx.hip and sim_mx.hip stage
// their planes with them.
#pragma once
#include "circatt_common.h"

namespace circatt {
namespace dma {

typedef int i4v __attribute__((ext_vector_type(4)));
constexpr unsigned kRsrcWord3 = 0x00020000;  // raw buffer, 32-bit data
// byte offset past every buffer (buffers are shorter): loads from there give 0
constexpr int kOut = 0x7fffff00;
constexpr int64_t kMaxBytes = 0x7ffffe00;

__device__ __forceinline__ i4v dma_rsrc(const float *p, int bytes) {
    const uint64_t b = reinterpret_cast<uint64_t>(p);
    return i4v{(int)(uint32_t)b, (int)((b >> 32) & 0xffffu), bytes, (int)kRsrcWord3};
}
// 16-byte LDS-DMA load: each active lane's four floats from byte voff + soff of
// the buffer to LDS byte m0 + 16 lane.  The caller waits (vmcnt(0) and a
// barrier).
__device__ __forceinline__ void dma16(i4v rs, unsigned m0, int voff, int soff) {
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
                 :
                 : "v"(voff), "s"(rs), "s"(soff), "{m0}"(m0)
                 : "memory");
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const float *p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p), (short)0, bytes, kRsrcWord3);
}

// v mod n for v in [-n, 2 n) (an integer remainder expands into some 35 vector
// instructions)
__device__ __forceinline__ int wrap(int v, int n) {
    v += v < 0 ? n : 0;
    return v - (v >= n ? n : 0);
}

}  // namespace dma
}  // namespace circatt
