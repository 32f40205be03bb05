// Loads that go from memory straight into LDS, for kernels that fill one buffer while they read another.
#pragma once
#include "common.h"

typedef __attribute__((address_space(3))) unsigned char lds_byte_t;

// 1 KB from memory into LDS, 16 bytes a lane from the lane's own address, or from `base` plus the lane's own offset; the place is
// the same for all lanes.  Written out because the compiler makes every LDS read wait for loads of this kind that are under way,
// also where they fill another buffer; lds_wait_and_meet waits for them instead.  (s_nop: the place register must rest a cycle
// before it is read.)
__device__ __forceinline__ void lds_bring(uint32_t place, const bf16_t* src) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(place), "v"(src) : "memory", "m0");
}
__device__ __forceinline__ void lds_bring_from(uint32_t place, uint32_t at, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(place), "v"(at), "s"(base) : "memory", "m0");
}
// the same for memory that this launch reads once or nearly so: it is the first to leave the caches
__device__ __forceinline__ void lds_bring_once_from(uint32_t place, uint32_t at, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(place), "v"(at), "s"(base) : "memory", "m0");
}
// all but the wavefront's N youngest loads are in, its LDS reads are through; then all wavefronts meet
template <int N = 0>
__device__ __forceinline__ void lds_wait_and_meet() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory"); }
