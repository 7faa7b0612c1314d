// Loads straight into LDS, and the waits that go with them (gfx950).
//
// Such a load ends when its data lies in LDS: `wait_loads` and then a barrier before another wavefront reads it.  They are
// written in assembly, as are the waits, so that which reads of LDS wait for which of them is what the kernels say and not what
// the compiler makes of it; they have no result in registers that could be taken for there before it is, and nothing of them
// may be on its way when a kernel ends.  Loads of a wavefront end in the order in which they were issued,
// the compiler's own among them (which it waits for as if these were not there, so at worst for more than it needs).
#pragma once

#include "common.h"

// 16 bytes a lane to lds + dst + 16 * lane; dst (bytes) the same for all lanes, and so `base` where the lanes' places are given
// as 32-bit offsets from it.  NT: past the caches.
template <bool NT>
__device__ __forceinline__ void lds_load16(void* lds, unsigned dst, unsigned offset, const void* base) {
  const unsigned at = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds)) + dst;
  if constexpr (NT)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(at), "v"(offset), "s"(base) : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(at), "v"(offset), "s"(base) : "memory", "m0");
}
template <bool NT>
__device__ __forceinline__ void lds_load16(void* lds, unsigned dst, const void* from) {
  const unsigned at = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds)) + dst;
  if constexpr (NT)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(at), "v"(from) : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(at), "v"(from) : "memory", "m0");
}
// 4 bytes a lane to lds + dst + 4 * lane.
__device__ __forceinline__ void lds_load4(void* lds, unsigned dst, unsigned offset, const void* base) {
  const unsigned at = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds)) + dst;
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(at), "v"(offset), "s"(base) : "memory", "m0");
}
// Until at most N of this wavefront's loads are on their way.
template <int N>
__device__ __forceinline__ void wait_loads() {
  static_assert(N >= 0 && N < 64, "what the counter holds");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// A barrier that leaves loads on their way alone; what this wavefront has read from LDS or written there itself is done.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
