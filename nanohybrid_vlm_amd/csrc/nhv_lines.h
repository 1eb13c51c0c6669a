// Memory to LDS by whole waves, for kernels that keep account of their loads themselves.
#pragma once
#include "nhv_common.h"

typedef __attribute__((address_space(3))) void* nhv_lds_ptr;

__device__ __forceinline__ uint32_t nhv_lds_address(const void* p) { return (uint32_t)(uintptr_t)(nhv_lds_ptr)p; }

// 16 bytes a lane from `from` to LDS at `to` + 16 lane (`to`: the same in the whole wave). Written as an instruction: of the
// builtin's loads the compiler keeps account, and waits for all of them before it reads any of the LDS that they may go to.
// ONCE: the line is read by nobody else, it passes the caches by.
template <bool ONCE>
__device__ __forceinline__ void nhv_load_to_lds(uint32_t to, const void* from) {
  to = __builtin_amdgcn_readfirstlane(to);
  if (ONCE) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(to), "v"(from) : "memory", "m0");
  else asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(to), "v"(from) : "memory", "m0");
}

// All of this wave's loads but the `YOUNGER` last ones have arrived, and it has read what it asked LDS for; behind the barrier
// that holds for every wave of the block.
template <int YOUNGER>
__device__ __forceinline__ void nhv_wait_and_meet() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(YOUNGER) : "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// A block goes over the inner dimension's chunks from a place of its own, round the end: were all blocks at the same columns at once,
// rows a power of two apart would all lie in a few of the caches' and the memory's channels, and so would the rows of x that all
// blocks read: gated products of 12,288 outputs and 4,096 columns at 64, 32 and 17 rows 45.8, 43.2 and 42.7 us without and 41.0, 38.0 and
// 37.8 with it; 6,144 of 4,096 at 1 to 16 rows 12.3 to 15.7 us, by where x happens to lie, and 11.7 to 12.6.
// (Rows of other lengths lie apart already, and the turning costs what it changes in what the caches hold: gated 9,728 of 2,560 at 1
// row 21.8 us without, 22.5 with it.)
// The order of an output's sum then hangs on the block that makes it: equal rows of w give results that differ by rounding. Logits,
// between which a choice is made, are summed so that they do not (gemm_fewrows_bf16.hip).
__device__ __forceinline__ int nhv_first_chunk(int block, int chunks, int K) {
  if (K % 2048) return 0;
  return (block / 8 + block % 8 * chunks / 8) % chunks;              // (blocks go to the 8 XCDs in turn)
}
// The i-th chunk from there; behind the last one, it again.
__device__ __forceinline__ int nhv_chunk(int first, int i, int chunks) {
  const int c = first + min(i, chunks - 1);
  return c < chunks ? c : c - chunks;
}
