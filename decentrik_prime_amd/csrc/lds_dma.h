// LDS DMA (global_load_lds_*) of the attention and GEMM kernels: loads from global memory straight
// into LDS, written as inline assembly so that the compiler does not guard every later LDS read
// with a wait for them; the kernels track these loads themselves with vmcnt waits.
//
// M0 holds the LDS address; it is saved and restored around each load.  gfx950 wants one wait state
// between a scalar write of M0 and an LDS-DMA instruction that reads it, which the compiler sees to
// for its own code but not inside an asm block: without the s_nop a load may take the old M0 and
// land at a stale LDS address.  (tests/test_wait_states.py reads the built library for it.)
#pragma once

#include "dk_common.h"

namespace dk {

// The LDS byte address of a pointer into shared memory.
__device__ __forceinline__ unsigned lds_addr(const void* p) {
  return (unsigned)(size_t)(__attribute__((address_space(3))) const void*)p;
}

// 16 bytes per lane from global memory into LDS at lds + 16 * lane.  The SADDR form: the global
// address is a wave-uniform 64-bit base held in SGPRs plus a 32-bit unsigned byte offset per lane.
// One address register per lane instead of two and no per-load vector arithmetic (the base advances
// from step to step in scalar registers): in a microbenchmark of the GEMM's main loop on MI355X the
// loads cost 12.5 % of the MFMA issue cycles in this form against 20 % with a 64-bit address per
// lane.
__device__ __forceinline__ void dma16s(uint64_t base, unsigned off, unsigned lds) {
  unsigned saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %1\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %2, %3\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved)
      : "s"(lds), "v"(off), "s"(base)
      : "memory");
}

// 4 bytes per lane from global memory (an address per lane) into LDS at lds + 4 * lane.
__device__ __forceinline__ void dma4(const void* src, unsigned lds) {
  unsigned saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %1\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dword %2, off\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved)
      : "s"(lds), "v"(src)
      : "memory");
}

// A wave-uniform 64-bit value in scalar registers.  readfirstlane returns int: each half goes
// through uint32_t so that the low half is zero-extended.
__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
  return ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((unsigned)(v >> 32)) << 32) |
         (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((unsigned)v);
}

// Wait until at most N of this wave's vector-memory instructions are in flight.
template <int N>
__device__ __forceinline__ void wait_vmem() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

}  // namespace dk
