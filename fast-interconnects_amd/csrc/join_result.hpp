// The sums of a join over its blocks.
#pragma once

#include "common.hpp"
#include "internal.hpp"
#include "pipeline.hpp"

namespace fij {

// Sums over the block, in thread 0 (red: [3][waves]); ends with a barrier.
template <uint32_t BLOCK>
__device__ __forceinline__ void block_sums(uint64_t (*red)[BLOCK / kWave], uint64_t& cnt, uint64_t& sb, uint64_t& sp) {
  const uint32_t w = threadIdx.x / kWave;
  cnt = wave_broadcast_last(wave_inclusive_scan(cnt));
  sb = wave_broadcast_last(wave_inclusive_scan(sb));
  sp = wave_broadcast_last(wave_inclusive_scan(sp));
  if (lane_id() == 0) {
    red[0][w] = cnt;
    red[1][w] = sb;
    red[2][w] = sp;
  }
  __syncthreads();
  cnt = sb = sp = 0;
  if (threadIdx.x == 0)
    for (uint32_t i = 0; i < BLOCK / kWave; ++i) {
      cnt += red[0][i];
      sb += red[1][i];
      sp += red[2][i];
    }
  __syncthreads();
}

// Ends a join whose blocks each hold sums of their own: the last block to get
// here adds up the blocks' sums in *result (true in that block).  partial
// [gridDim.x] is scratch, done [kDoneWords] counts blocks and is zero between
// joins: one counter after the other serves its blocks, so those of a large
// grid count in groups and the last of a group for all of it.  A
// launch of its own for the sum takes 4 us of device time.  The sums travel by
// device-scope atomics, complete before the block is counted: a __threadfence
// per block instead writes back its die's L2 each time, which made a served
// request's 512 blocks 15 us slower.
template <uint32_t BLOCK>
__device__ __forceinline__ bool finish_join(JoinAggregate* partial, uint32_t* done, JoinAggregate* result,
                                            uint64_t (*red)[BLOCK / kWave], uint32_t* s_last, uint64_t cnt,
                                            uint64_t sb, uint64_t sp) {
  block_sums<BLOCK>(red, cnt, sb, sp);
  if (gridDim.x > 1) {
    if (threadIdx.x == 0) {
      uint64_t* const r = reinterpret_cast<uint64_t*>(partial + blockIdx.x);
      __hip_atomic_exchange(r, cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_exchange(r + 1, sb, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_exchange(r + 2, sp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      bool last = true;
      uint32_t n = gridDim.x;
      if (n > 4 * kDoneGroups) {
        const uint32_t g = blockIdx.x % kDoneGroups;
        uint32_t* const group = done + (g + 1) * kDoneStride;
        last = atomicAdd(group, 1u) == (n - g + kDoneGroups - 1) / kDoneGroups - 1;
        if (last) *group = 0;
        n = kDoneGroups;
      }
      *s_last = last && atomicAdd(done, 1u) == n - 1 ? 1u : 0u;
    }
    __syncthreads();
    if (!*s_last) return false;  // uniform
    cnt = sb = sp = 0;
    for (uint32_t i = threadIdx.x; i < gridDim.x; i += BLOCK) {
      const uint64_t* r = reinterpret_cast<const uint64_t*>(partial + i);
      cnt += __hip_atomic_load(r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      sb += __hip_atomic_load(r + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      sp += __hip_atomic_load(r + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    block_sums<BLOCK>(red, cnt, sb, sp);
    if (threadIdx.x == 0) *done = 0;
  }
  if (threadIdx.x == 0) *result = JoinAggregate{cnt, sb, sp};
  return true;
}

}  // namespace fij
