// Rows of a matrix as operands of 16x16 matrix instructions, through LDS.  An operand lies with a row in every lane, neighbouring lanes in
// different rows; loaded that way from memory, a load of 1 KiB takes the unit that takes addresses 64 cycles (a lane a cycle; measured for
// every tile of the float32 product, 16 bytes a cycle for a whole compute unit).  Direct loads with eight lanes to a row's 128 bytes
// take 16, and reading the operand back from LDS 8.  A wavefront has stages of its own: it waits for its own loads and meets no barrier.
//
// A block is 16 rows of 128 bytes (2 KiB): two loads of eight rows.  What stands c-th in a row r lies in place c ^ (r & 7).  A read of 16 bytes a lane
// takes its lanes sixteen at a time, but not in their order: rows 0 to 3 and 12 to 15 of one operand piece go with rows 4 to 11 of the next
// quarter's.  Those meet in no bank if the quarters of a wavefront read neighbouring places: pieces q and q + 4 by quarter q, 1.8 ns a read
// of a unit (linear 1.8).  Pieces 2 q and 2 q + 1, two halves of 16 consecutive k, took 3.4 from places 2 q and 2 q + 1; where an operand is such a
// pair the loads put piece 2 q into place q and piece 2 q + 1 into place q + 4 (piece_of).
#pragma once
#include <hip/hip_runtime.h>

// the piece of a row's eight that stands c-th where a lane's operand is pieces 2 q and 2 q + 1
__device__ __forceinline__ int piece_of(int c) { return ((c & 3) << 1) | (c >> 2); }

// s_waitcnt with only vmcnt set (gfx9 encoding: vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] | vmcnt[5:4] << 14)
template <int N> __device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N <= 63, "vmcnt counts to 63");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// N blocks have arrived in registers when this returns.  x, y: LDS byte addresses of this lane's two pieces of the first; E has two members
// x, y of 16 bytes
template <int N, class E> __device__ __forceinline__ void read_some_blocks(E* e, unsigned x, unsigned y) {
  static_assert(N >= 1 && N <= 4, "up to eight reads at a time");
  if constexpr (N == 1)
    asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(e[0].x), "=&v"(e[0].y) : "v"(x), "v"(y) : "memory");
  if constexpr (N == 2)
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %4 offset:2048\n\tds_read_b128 %3, %5 offset:2048\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(e[0].x), "=&v"(e[0].y), "=&v"(e[1].x), "=&v"(e[1].y) : "v"(x), "v"(y) : "memory");
  if constexpr (N == 3)
    asm volatile("ds_read_b128 %0, %6\n\tds_read_b128 %1, %7\n\tds_read_b128 %2, %6 offset:2048\n\tds_read_b128 %3, %7 offset:2048\n\t"
                 "ds_read_b128 %4, %6 offset:4096\n\tds_read_b128 %5, %7 offset:4096\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(e[0].x), "=&v"(e[0].y), "=&v"(e[1].x), "=&v"(e[1].y), "=&v"(e[2].x), "=&v"(e[2].y)
                 : "v"(x), "v"(y) : "memory");
  if constexpr (N == 4)
    asm volatile("ds_read_b128 %0, %8\n\tds_read_b128 %1, %9\n\tds_read_b128 %2, %8 offset:2048\n\tds_read_b128 %3, %9 offset:2048\n\t"
                 "ds_read_b128 %4, %8 offset:4096\n\tds_read_b128 %5, %9 offset:4096\n\tds_read_b128 %6, %8 offset:6144\n\t"
                 "ds_read_b128 %7, %9 offset:6144\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(e[0].x), "=&v"(e[0].y), "=&v"(e[1].x), "=&v"(e[1].y), "=&v"(e[2].x), "=&v"(e[2].y), "=&v"(e[3].x), "=&v"(e[3].y)
                 : "v"(x), "v"(y) : "memory");
}
template <int BLOCKS, class E> __device__ __forceinline__ void read_blocks(E* e, unsigned x, unsigned y) {
  constexpr int R = BLOCKS % 4;
#pragma unroll
  for (int b = 0; b + 4 <= BLOCKS; b += 4) read_some_blocks<4>(e + b, x + b * 2048, y + b * 2048);
  if constexpr (R) read_some_blocks<(R ? R : 1)>(e + BLOCKS - R, x + (BLOCKS - R) * 2048, y + (BLOCKS - R) * 2048);
}

// A step's loads, 2 BLOCKS of them, are back; those of the `behind` steps asked for after it may still be out.
template <int BLOCKS, int STAGES> __device__ __forceinline__ void wait_for_step(int behind) {      // the same in every lane
  if (STAGES >= 4 && behind == 3) wait_vmcnt<STAGES >= 4 ? 6 * BLOCKS : 0>();
  else if (STAGES >= 3 && behind == 2) wait_vmcnt<STAGES >= 3 ? 4 * BLOCKS : 0>();
  else if (STAGES >= 2 && behind == 1) wait_vmcnt<STAGES >= 2 ? 2 * BLOCKS : 0>();
  else wait_vmcnt<0>();
}

// A wavefront's steps: load(step, stage's byte) asks for the 2 BLOCKS loads of a step, multiply(blocks) takes them when they are in
// registers.  x, y: as above, in stage 0.  A stage is asked for again as soon as it has been read.
template <int BLOCKS, int STAGES, class E, class Load, class Multiply>
__device__ __forceinline__ void staged_steps(int steps, unsigned x, unsigned y, Load load, Multiply multiply) {
  static_assert(STAGES >= 1 && STAGES <= 4, "up to four stages");
#pragma unroll
  for (int d = 0; d < STAGES; ++d)
    if (d < steps) load(d, d * BLOCKS * 2048);
  unsigned stage = 0;
  for (int i = 0; i < steps; ++i) {
    wait_for_step<BLOCKS, STAGES>(min(STAGES, steps - i) - 1);
    E e[BLOCKS];
    read_blocks<BLOCKS>(e, x + stage, y + stage);
    if (i + STAGES < steps) load(i + STAGES, stage);
    __builtin_amdgcn_sched_barrier(0);
    multiply(e);
    stage = stage == (STAGES - 1) * BLOCKS * 2048 ? 0 : stage + BLOCKS * 2048;
  }
}
