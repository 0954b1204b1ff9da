// Direct global -> LDS loads and the waits and barriers of the pipelined k-loops that use them,
// shared by the 16-bit and the f32 GEMM kernels (gfx950 only).
#pragma once

#include "device.hpp"

// buffer_load_dwordx4 ... lds: a direct global -> LDS load (LDS address from M0, lane l at + 16 l)
// whose global address is a buffer resource (scalar) plus a per-lane 32-bit offset and a scalar
// offset; offsets past the resource's size read 0. The LLVM intrinsic behind it is bound by name,
// outside any namespace so that the declaration keeps external linkage.
typedef int i32x4 __attribute__((ext_vector_type(4)));
__device__ void raw_buffer_load_lds(i32x4 rsrc, __attribute__((address_space(3))) void* lds, int size, int voffset,
                                    int soffset, int offset, int aux) __asm("llvm.amdgcn.raw.buffer.load.lds");

namespace s1 {

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Workgroup barrier without the memory fence of __syncthreads: the fence would make the compiler
// drain every outstanding global->LDS load (vmcnt(0)) at each k-tile and serialise the pipeline.
// The "memory" clobber keeps LDS accesses on their side of it; completion of the async loads is
// awaited explicitly with wait_vmcnt before it.
__device__ __forceinline__ void barrier_lds() { asm volatile("s_barrier" ::: "memory"); }

// Raw buffer resource over [p, p + bytes): base address, no stride, the byte count, and the third
// dword of every gfx9 buffer resource (32-bit data format, no swizzle).
__device__ __forceinline__ i32x4 buffer_rsrc(const void* p, uint32_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  i32x4 r;
  r.x = __builtin_amdgcn_readfirstlane(int(uint32_t(a)));
  r.y = __builtin_amdgcn_readfirstlane(int(uint32_t(a >> 32) & 0xffff));
  r.z = __builtin_amdgcn_readfirstlane(int(bytes));
  r.w = 0x00020000;
  return r;
}

// 16 bytes per lane from rsrc + voff + soff to the KiB of LDS at `lds` (a generic LDS pointer).
__device__ __forceinline__ void load16_lds(i32x4 rsrc, char* lds, int voff, int soff) {
  raw_buffer_load_lds(rsrc, reinterpret_cast<__attribute__((address_space(3))) void*>(uint32_t(reinterpret_cast<uintptr_t>(lds))),
                      16, voff, soff, 0, 0);
}

// Wait until at most `ahead` k-tiles of this wave's loads (LPW loads each) are in flight.
template <int LPW, int MAXA>
__device__ __forceinline__ void wait_ahead(int ahead) {
  if constexpr (MAXA > 0) {
    if (ahead >= MAXA) {
      wait_vmcnt<MAXA * LPW>();
      return;
    }
    wait_ahead<LPW, MAXA - 1>(ahead);
  } else {
    wait_vmcnt<0>();
  }
}

}  // namespace s1
