// lds_dma.hpp -- memory straight into LDS, 16 bytes per lane, and the waits that go with it.
#pragma once
#include "devutil.hpp"

namespace crabml_hip {

__device__ __forceinline__ unsigned lds_address(const void* l) {
  return (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(size_t)(const __attribute__((address_space(3))) void*)l);
}
// 16 bytes per lane from memory into LDS at the address `at` + 16 lane (wave-uniform).  As assembly, because the compiler would wait for ALL of them
// in front of the next LDS read (it cannot tell the buffers apart); who waits for what is landed_barrier's business.
// (m0, the LDS address of such a load, needs one wait state behind its write; nothing else here uses it.)
__device__ __forceinline__ void lds_dma16(const void* g, unsigned at) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(at) : "memory");
}
// the same from `off` bytes behind a wave-uniform base
__device__ __forceinline__ void lds_dma16(const void* base, unsigned off, unsigned at) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(at) : "memory");
}
// waits until at most N of this wave's memory requests are outstanding, then for the workgroup.  (__syncthreads would drain them all.)
template <int N>
__device__ __forceinline__ void landed_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

}  // namespace crabml_hip
