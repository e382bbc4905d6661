// tl_lds.h — device helpers shared by kernels that move tiles straight from memory to LDS (tl_dense.hip, tl_hattn.hip).
#pragma once
#include <hip/hip_runtime.h>

// 16 bytes a lane from base + off to LDS bytes at .. at + 1023, no registers in between (at, base: the same in all lanes). M0 holds the
// LDS address and belongs to the compiler: saved and restored in the same statement
__device__ __forceinline__ void tl_lds_load16(unsigned at, unsigned off, const void* base) {
  unsigned keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "s"(at), "v"(off), "s"(base) : "memory");
}
// ... 4 bytes a lane to LDS bytes at .. at + 255
__device__ __forceinline__ void tl_lds_load4(unsigned at, unsigned off, const void* base) {
  unsigned keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %2, %3\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "s"(at), "v"(off), "s"(base) : "memory");
}
// an address that is the same in all lanes, in scalar registers
template <class T>
__device__ __forceinline__ const T* tl_uniform(const T* p) {
  const unsigned long long a = reinterpret_cast<unsigned long long>(p);
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)a), hi = __builtin_amdgcn_readfirstlane((unsigned)(a >> 32));
  return reinterpret_cast<const T*>((unsigned long long)hi << 32 | lo);
}
// all but the last N of this wave's loads have arrived, and every wave of the workgroup is here
template <int N>
__device__ __forceinline__ void tl_lds_barrier() {
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory");
}
