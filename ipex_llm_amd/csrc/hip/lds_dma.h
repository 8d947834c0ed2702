// LDS-DMA of the tile kernels: buffer_load_dwordx4 ... lds, 16 bytes a lane straight from memory to LDS (a wave-uniform
// base + lane * 16), no register in between.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace illm {

typedef int32_t dma_rsrc __attribute__((ext_vector_type(4)));

// buffer descriptor: base, num_records = bytes (reads past it return 0)
__device__ __forceinline__ dma_rsrc make_dma_rsrc(const void* base, uint32_t bytes) {
  const uint64_t p = (uint64_t)(uintptr_t)base;
  return dma_rsrc{(int32_t)(uint32_t)p, (int32_t)((uint32_t)(p >> 32) & 0xffffu), (int32_t)bytes, 0x00020000};
}

// LDS byte address of a wave-uniform pointer
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const __attribute__((address_space(3))) uint8_t*)p);
}

// Issued from inline asm ON PURPOSE: hipcc cannot tell these LDS writes from the reads of another buffer and would drain
// vmcnt(0) before each of those; the caller's own s_waitcnt and barrier order them.  A write of m0 needs one wait state
// before the LDS-DMA that reads it, which hipcc does not add inside asm.
__device__ __forceinline__ void lds_dma16(const dma_rsrc& rs, uint32_t lds, uint32_t voff, int soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :: "s"(lds), "v"(voff), "s"(rs), "s"(soff) : "memory", "m0");
}
__device__ __forceinline__ void lds_dma16(const dma_rsrc& rs, uint32_t lds, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               :: "s"(lds), "v"(voff), "s"(rs) : "memory", "m0");
}

}  // namespace illm
