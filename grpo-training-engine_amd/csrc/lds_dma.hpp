// Loads straight to LDS and waits for them by count (gfx950).
//
// The kernels that use these keep several stages of loads in flight in one LDS
// ring. The loads are volatile asm without results, and every wait is explicit: the
// compiler, which does not tell the ring's stages apart, would wait for all
// outstanding loads before each LDS read. Its own waits for its own loads stay
// correct, since loads retire in order and it only undercounts what is outstanding
// (it then waits for more than it needs, never for less). m0, which carries the LDS
// address, is a reserved register: it cannot be named as clobbered, and the compiler sets
// it anew before each instruction of its own that reads it.
#pragma once

#include "common.hpp"

namespace grpo {

// 16 bytes per lane from base + voff to 1 KiB at the wave-uniform LDS address lds.
__device__ __forceinline__ void dma16(uint32_t lds, uint32_t voff, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds),
               "v"(voff), "s"(base)
               : "memory");
}

// 4 bytes per lane from base + voff to 256 bytes at lds.
__device__ __forceinline__ void dma4(uint32_t lds, uint32_t voff, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds),
               "v"(voff), "s"(base)
               : "memory");
}

// Wait until at most N vector memory operations are outstanding.
template <int N>
__device__ __forceinline__ void wait_vm() {
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}
// ... and every LDS operation is done.
template <int N>
__device__ __forceinline__ void wait_vm_lds() {
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | ((N >> 4) << 14));
}

__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)p;
}

}  // namespace grpo
