// LDS-direct loads (gfx950 `buffer_load ... lds`) and the waits and barriers
// that go with them.
#pragma once

#include "aexq_device.hpp"

namespace aexq {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(1))) char gchar;  // global memory
typedef __attribute__((address_space(1))) f32x4 gf32x4;
typedef __attribute__((address_space(1))) u32x4 gu32x4;

// LDS byte address of a generic pointer into LDS (the low half of the
// generic address), wave-uniform.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)p);
}

// One LDS-direct load: lane i's BYTES (16 or 4) at byte voff of resource r go
// to LDS byte lds + BYTES * i; offsets past the resource's end write zeros.
// Written as assembly so that the compiler does not see LDS stores in flight:
// it would otherwise wait for every outstanding load before each LDS read.
// The kernel orders them itself -- s_waitcnt vmcnt for its own loads, then a
// barrier for the other waves' -- and the memory clobber keeps the compiler
// from moving LDS accesses across a load.
template <int BYTES>
__device__ __forceinline__ void dma(__amdgpu_buffer_rsrc_t r, uint32_t lds, uint32_t voff) {
  static_assert(BYTES == 16 || BYTES == 4, "dword or dwordx4");
  if constexpr (BYTES == 16)
    asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                 :
                 : "s"(lds), "v"(voff), "s"(r)
                 : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dword %1, %2, 0 offen lds"
                 :
                 : "s"(lds), "v"(voff), "s"(r)
                 : "memory", "m0");
}

// s_waitcnt vmcnt(N) with the other counters left alone (gfx9 encoding).
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | 0x70 | 0xF00 | ((N >> 4) << 14));
}
// s_waitcnt lgkmcnt(0).
__device__ __forceinline__ void wait_lgkm0() { __builtin_amdgcn_s_waitcnt(0xC07F); }
// Workgroup barrier without the fence __syncthreads() adds (whose vmcnt(0)
// would also wait for the LDS-direct loads of the steps ahead); the empty asm
// statements keep the compiler from moving LDS accesses across it.
__device__ __forceinline__ void bar() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Waits until the loads of at most min(KMAX, ahead) steps (NL instructions
// each) are outstanding, the older ones landed; `ahead` is wave-uniform.
template <int NL, int KMAX>
__device__ __forceinline__ void wait_steps(int ahead) {
  if constexpr (KMAX > 0) {
    if (ahead >= KMAX)
      wait_vm<KMAX * NL>();
    else
      wait_steps<NL, KMAX - 1>(ahead);
  } else {
    wait_vm<0>();
  }
}

}  // namespace aexq
