// Loads that write into LDS themselves, with waits counted by hand: what the kernels that keep several stages on their way share.
// A plain barrier behind a counted wait lets the stages that are still wanted stay in flight, where __syncthreads() would wait for all of them.
#pragma once
#include "common.h"

// until at most ``n`` of this wave's vector loads are still on their way; until its LDS reads are done
#define TILE_WAIT_LOADS(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | (((n) >> 4) << 14) | (7 << 4) | (15 << 8))
#define TILE_WAIT_LDS() __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4))
#define TILE_BARRIER()             \
  do {                             \
    asm volatile("" ::: "memory"); \
    __builtin_amdgcn_s_barrier();  \
    asm volatile("" ::: "memory"); \
  } while (0)

[[maybe_unused]] static __device__ const int4 tile_zeros = {0, 0, 0, 0};  // what stands for a piece beyond K
