// Global memory -> LDS loads without registers, and the waits of a ring of LDS buffers fed by
// them (the tile product of gemm_f16.hip).
#pragma once

#include "common.h"

namespace relay_hip {

// buffer_load_dwordx4 ... lds: lane l's 16 bytes go to LDS address m0 + 16 l. Written as
// asm because the builtin makes the compiler wait for vmcnt(0) before every LDS read it
// cannot tell apart from the destination; here the ring's own waits (wait_vm) order them.
// The instruction has no output register; every offset is clamped to the matrix.
__device__ __forceinline__ uint4v lds_rsrc(const void* base) {
  const uint64_t p = reinterpret_cast<uint64_t>(base);
  return uint4v{static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(p))),
                static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(p >> 32))) & 0xffffu,
                0x7fffffffu, 0x00020000u};
}

__device__ __forceinline__ void load_to_lds(uint4v rsrc, uint32_t voffset, uint32_t soffset, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
               :
               : "v"(voffset), "s"(rsrc), "s"(soffset), "s"(lds)
               : "memory");
}

// At most N of this wave's vector-memory operations still outstanding.
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

// wait_vm<P * later> for later = min(later, MAX) (the count is an immediate).
template <int P, int MAX>
__device__ __forceinline__ void wait_stages(int later) {
  if constexpr (MAX == 0) {
    wait_vm<0>();
  } else {
    if (later >= MAX)
      wait_vm<P * MAX>();
    else
      wait_stages<P, MAX - 1>(later);
  }
}

// A workgroup barrier after which LDS contents written by any wave's landed loads are visible,
// and no LDS access moves across it.
__device__ __forceinline__ void ring_barrier() {
  asm volatile("" : : : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" : : : "memory");
}

__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const char*)p));
}

}  // namespace relay_hip
