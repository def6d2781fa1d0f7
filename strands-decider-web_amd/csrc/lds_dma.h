// LDS DMA written out, gfx950: the compiler would otherwise wait for every DMA in flight before any LDS read, and for
// the loads issued after it too. Lane l's bytes, from base + voff, land at lds + 16 l (dwordx4) or lds + 4 l (dword); the
// kernel's own waits (vmcnt) order them. m0, the DMA's LDS base, is a register the compiler reserves and does not preserve
// across asm: sound while no compiler-generated code of the kernels that use these keeps a value in it (tests/test_strip_guards.py checks
// the assembly).
#pragma once
#include <hip/hip_runtime.h>

namespace ha {
namespace {

__device__ __forceinline__ void dma16(unsigned lds, unsigned voff, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(__builtin_amdgcn_readfirstlane(lds)),
               "v"(voff), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void dma4(unsigned lds, unsigned voff, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, %2" ::"s"(__builtin_amdgcn_readfirstlane(lds)),
               "v"(voff), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ unsigned lds_addr(const void* p) {
  return (unsigned)(size_t)(const __attribute__((address_space(3))) char*)p;
}

}  // namespace
}  // namespace ha
