// Loads that write LDS directly, for the kernels that move whole tiles that way.
#pragma once

#include "common.hpp"

namespace npamd {

// A pointer that is the same in every lane, said so to the compiler (an "s" operand has to live in scalar registers).
__device__ __forceinline__ const uint8_t* uniform_ptr(const uint8_t* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return reinterpret_cast<const uint8_t*>(((uint64_t)hi << 32) | lo);
}

// Lane l's 16 (4) bytes land at dst + 16 l (4 l); dst is uniform over the wave.  The statements write m0, which the compiler does not
// let an asm statement declare as clobbered; that is sound as long as the compiler keeps nothing of its own in m0 in the kernels
// that use them, which the tests of the generated code check.  Nothing but waits and scheduling barriers keeps a transfer behind reads of the
// place it fills.
__device__ __forceinline__ void lds_load16(uint32_t dst, uint32_t voff, const void* base) {
  dst = __builtin_amdgcn_readfirstlane(dst);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(voff), "s"(base) : "memory");
}
__device__ __forceinline__ void lds_load4(uint32_t dst, uint32_t voff, const void* base) {
  dst = __builtin_amdgcn_readfirstlane(dst);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(dst), "v"(voff), "s"(base) : "memory");
}

}  // namespace npamd
