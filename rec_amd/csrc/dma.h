// Direct loads from memory into LDS (gfx950 global_load_lds), untracked by the
// compiler.
#pragma once

#include "common.h"

namespace rec {

// Direct loads into LDS: lane i's 16 (4) bytes at p + voff arrive at lds + 16 i
// (4 i).  Not tracked by the compiler: dma_wait() before the barrier in front
// of the first read.
__device__ __forceinline__ void dma16(uint32_t lds, const char* p, uint32_t voff) {  // p the same in every lane
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff), "s"(p) : "memory");
}
__device__ __forceinline__ void dma16(uint32_t lds, const uint8_t* p) {  // p the lane's own
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(p) : "memory");
}
__device__ __forceinline__ void dma4(uint32_t lds, const char* p, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(voff), "s"(p) : "memory");
}
__device__ __forceinline__ void dma_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// A pointer that is the same in every lane, for a scalar register pair.
__device__ __forceinline__ const char* uniform_ptr(const void* p) {
  const uint64_t u = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u), hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
  return (const char*)(((uint64_t)hi << 32) | lo);
}

// The LDS byte address of a shared variable.
template <typename T>
__device__ __forceinline__ uint32_t lds_address(T& x) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)&x;
}

}  // namespace rec
