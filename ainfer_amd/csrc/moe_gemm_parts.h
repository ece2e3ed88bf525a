// moe_gemm_parts.h - device pieces shared by the grouped expert GEMMs
// (moe_gemm.hip, moe_gemm_w4a8.hip) and the router GEMM: global->LDS DMA with
// scalar bases, the ring's waits and barrier, the weight rows' swizzle.
#pragma once
#include "moe_common.h"

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ void dma16(const void *g, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
               :
               : "v"(g), "s"(lds_addr)
               : "memory", "m0");
}

// The same with a scalar base address (sbase64) and a 32-bit per-lane offset.
__device__ __forceinline__ void dma16s(uint32_t off, uint64_t base, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(off), "s"(base), "s"(lds_addr)
               : "memory", "m0");
}
// one dword per lane
__device__ __forceinline__ void dma4s(uint32_t off, uint64_t base, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
               :
               : "v"(off), "s"(base), "s"(lds_addr)
               : "memory", "m0");
}
// a wave-uniform address in SGPRs
__device__ __forceinline__ uint64_t sbase64(const void *p) {
  const uint64_t b = (uint64_t)(uintptr_t)p;
  return (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b) |
         ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(b >> 32)) << 32);
}

template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

// Every LDS read this wave issued completes before the barrier: s_barrier
// alone does not wait for them, and the compiler is free to place the
// lgkmcnt wait of a fragment read after the barrier (with the MFMA that uses
// it).  A wave past the barrier may then refill that ring stage by DMA while
// the read is still queued.  (Without this wait the router GEMM below read a
// refilled stage now and then: wrong approximate logits, wrong top-k.)
__device__ __forceinline__ void block_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// B chunk swizzle: 2-bit function of the row such that 8 consecutive rows
// (32 banks x 4 B) and 16 consecutive rows (64 banks) both land the 16-byte
// chunks of one logical column in distinct bank groups.
__device__ __forceinline__ int bswz(int r) {
  return (((r >> 1) ^ (r >> 3)) & 1) | (((r >> 2) & 1) << 1);
}

// sum over the 16 lanes of a DPP row (lane & 15), in every lane of the row
__device__ __forceinline__ float row16_sum(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, false));   // quad [1,0,3,2]
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, false));   // quad [2,3,0,1]
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xF, 0xF, false));  // half mirror
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xF, 0xF, false));  // row mirror
  return v;
}

}  // namespace
