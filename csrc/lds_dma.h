// Loads from global memory straight into LDS.
#pragma once
#include "common.h"

// 16 bytes a lane from base + off (both as the lane sees them; base uniform)
// to LDS byte `lds` (uniform) + 16 lane.  The compiler does not see these
// loads: whoever reads the bytes waits for vmcnt first, then for the other
// waves at a barrier.
__device__ __forceinline__ void load_to_lds(const void* base, u32 off,
                                            u32 lds) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %2"
      :
      : "s"(lds), "v"(off), "s"(base)
      : "memory", "m0");
}

// the same with 4 bytes a lane
__device__ __forceinline__ void load4_to_lds(const void* base, u32 off,
                                             u32 lds) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dword %1, %2"
      :
      : "s"(lds), "v"(off), "s"(base)
      : "memory", "m0");
}

// own loads have landed, everybody's after the barrier
__device__ __forceinline__ void lds_loads_done() {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
}

// own loads but the last N have landed, and reads of LDS are done; then
// everybody's
template <int N>
__device__ __forceinline__ void loads_but() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N)
               : "memory");
}

// Swizzle of rows of 2, 4, 8 or 16 16-byte slots: the slots of 16 consecutive
// rows at one column fall into different banks, and so do those of the two halves
// of 32 rows that a 16-byte read of a row a lane takes together (below).
template <int SLOTS>
__device__ __forceinline__ int slot_key(int row) {
  static_assert(SLOTS == 2 || SLOTS == 4 || SLOTS == 8 || SLOTS == 16, "");
  return SLOTS == 16  ? row & 15
         : SLOTS == 8 ? (row >> 1) & 7
         : SLOTS == 4 ? (row >> 2) & 3
                      : (row >> 3) & 1;
}

// Swizzle of rows of 4, 8 or 16 16-byte slots for reads of 16 bytes where lane
// group l4 reads slots l4 S / 4 ..: such a read takes 16 lanes at a time, lanes
// 0-3, 12-15, 20-27 and 4-11, 16-19, 28-31 (and so on from 32), and each of
// these sets finds its slots in different banks.
template <int S>
__device__ __forceinline__ int slot_key16(int row) {
  static_assert(S == 4 || S == 8 || S == 16, "");
  const int q = 0xD2 >> (row >> 1 & 6) & 3;      // 2 0 1 3 of row / 4
  return S == 4 ? q : (S == 8 ? q * 2 + (row >> 1 & 1) : q * 4 + (row & 3));
}
