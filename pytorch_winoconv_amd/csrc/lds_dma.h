#pragma once
#include "wc_common.h"

namespace wc {

// LDS-DMA: lane l of a wavefront brings the 16 bytes at byte `voff` of a buffer to LDS byte lds_addr + 16 l, without a register.  Offsets outside the
// descriptor's range (kOutside) bring zeros.  Inline assembly, since the compiler cannot know which LDS bytes such a load fills and would wait
// for all of them before every LDS read; the kernels count what may still be on its way.  Addresses are multiples of 16.
typedef uint32_t DmaDesc __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void dma16(DmaDesc desc, unsigned voff, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" :: "v"(voff), "s"(desc), "s"(lds_addr) : "memory");
}

// The buffer of `bytes` bytes at p; offsets have 31 bits
__device__ __forceinline__ DmaDesc dma_descriptor(const void* p, long long bytes) {
  const unsigned long long u = reinterpret_cast<unsigned long long>(p);
  const unsigned n = (unsigned)max(min(bytes, 0x7fffffffll), 0ll);
  return DmaDesc{(unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)u), (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(u >> 32)),
                 (unsigned)__builtin_amdgcn_readfirstlane((int)n), 0x00020000u};
}

}  // namespace wc
