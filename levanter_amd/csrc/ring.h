// k-tiles of 64 bfloat16 numbers a row (lines of 128 bytes) on their way from memory straight into LDS.
#pragma once
#include "common.h"

// Which of its line's eight 16-byte chunks a row keeps at place 0 of LDS (at place p: p ^ that). LDS has 64 banks, so 16 lanes' chunks (two rows' worth of banks) are
// served at once: 16 rows one behind the other (rows), or the 16 rows 8 q + r (r < 4) that an operand of eights of columns takes (columns), each have their own.
__device__ __forceinline__ int ring_swap_rows(int row) { return (row >> 1) & 7; }
__device__ __forceinline__ int ring_swap_columns(int row) { return ((row >> 1) & 1) | ((row >> 2) & 6); }

// 16 bytes a lane from base + off straight into LDS, at lds + 16 * lane. In assembly because the compiler waits for all such loads before any read of LDS; no
// register is written, and whoever reads the LDS waits for vmcnt (ring_wait) and a barrier first. m0 is reserved to the compiler, which keeps nothing in it from one
// instruction to the next and takes no clobber of it; the kernels here have no other instruction that reads it.
__device__ __forceinline__ void lines_to_lds(uint32_t lds, uint32_t off, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory");
}
// all but the wave's N youngest loads have landed
template <int N>
__device__ __forceinline__ void ring_wait() {
  static_assert(N >= 0 && N <= 63, "vmcnt counts to 63");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// all but the loads of the `newer` youngest k-tiles, L loads each, R k-tiles in the ring
template <int R, int L>
__device__ __forceinline__ void ring_wait_for(int newer) {
  switch (newer) {
    case 7: ring_wait<R >= 8 ? 7 * L : 0>(); break;
    case 6: ring_wait<R >= 7 ? 6 * L : 0>(); break;
    case 5: ring_wait<R >= 6 ? 5 * L : 0>(); break;
    case 4: ring_wait<R >= 5 ? 4 * L : 0>(); break;
    case 3: ring_wait<R >= 4 ? 3 * L : 0>(); break;
    case 2: ring_wait<2 * L>(); break;
    case 1: ring_wait<L>(); break;
    default: ring_wait<0>();
  }
}
__device__ __forceinline__ uint32_t lds_offset(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p;
}
