// Loads from global memory straight into LDS
#pragma once
#include "common.cuh"

namespace ffmoe {

// 16 (4) bytes per lane from base + offset into LDS at lds + 16 (4) x lane. No register holds the data, so the caller's
// s_waitcnt before the barrier that publishes the tile is all the bookkeeping there is. (m0 is a reserved register: nothing the
// compiler generates for these kernels reads it, and it accepts no clobber of it.)
__device__ __forceinline__ void lds_load16(uint32_t lds, uint64_t base, uint32_t offset) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(offset), "s"(base) : "memory");
}
// with the streaming hint: the line is the first the L2 gives up again
__device__ __forceinline__ void lds_load16_nt(uint32_t lds, uint64_t base, uint32_t offset) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(lds), "v"(offset), "s"(base) : "memory");
}
__device__ __forceinline__ void lds_load16(uint32_t lds, const void* p) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(p) : "memory");
}
__device__ __forceinline__ void lds_load4(uint32_t lds, const void* p) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(lds), "v"(p) : "memory");
}
__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return uint32_t(uni(int(uint32_t(uintptr_t((const __attribute__((address_space(3))) void*)p)))));
}

}  // namespace ffmoe
