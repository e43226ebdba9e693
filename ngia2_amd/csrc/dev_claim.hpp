// dev_claim.hpp -- what the binned alignment kernels share: the early-exit test
// and a wavefront's claim on its bin's work queue (device code).
#pragma once

#include "dev_common.hpp"

namespace ngia {

// Early exit.  The kernels compute the LCS of the band-masked match matrix
// (the bit-parallel update with the masks of words outside the band set to
// 0 is exactly the banded recurrence), and an LCS grows by at most one per
// target character; the pass test (buildGraph.hpp:248) is monotone in the
// LCS.  So a pair whose LCS after `done` characters, plus the characters left,
// fails the test scores 0 whatever follows.
__device__ inline bool cannot_pass(uint32_t lcs_now, uint32_t done, uint32_t R, uint32_t T,
                                   float thr) {
  const uint32_t left = T > done ? T - done : 0u;
  return lcs_score(lcs_now + left, R, T, thr) == 0u;
}

// A wavefront's claim on its bin's work queue.  Every pair taken through a
// per-pair atomic on one counter serialises a bin of many short pairs on that
// address, so one atomic claims `chunk` consecutive items of a slice and the
// wave hands them out in order.  The chunk follows the bin's size, so each
// wave still gets many claims and the queue drains evenly: count / (16
// waves' worth), between `lo` and `hi` (lo >= the most items handed out at
// once).  The wave starts on the slice of its XCD (kQueueSlices slices, one
// counter each) with the chunk of its number there, which needs no claim; the
// counters hand out what follows the waves' first chunks, so a queue that
// those cover is never touched.  When a slice is exhausted the wave reads the
// counters of the slices that have more and moves to the next one with items
// left; with none left the queue is drained.  All members are wave-uniform;
// take() is called by the whole wave at a convergent point.
struct WaveClaim {
  uint32_t next = 0, end = 0, chunk = 1, count, slice;
  bool drained = false;
  __device__ WaveClaim(uint32_t count_, uint32_t lo, uint32_t hi) : count(count_) {
    const uint32_t per = count / (gridDim.x * (blockDim.x / 64u) * 16u);
    chunk = per < lo ? lo : per > hi ? hi : per;
    slice = blockIdx.x % kQueueSlices;
    const uint32_t s0 = slice_lo(slice), len = slice_lo(slice + 1) - s0;
    const uint32_t first = blockIdx.x / kQueueSlices * chunk;
    if (first < len) {
      next = s0 + first;
      end = s0 + (len - first < chunk ? len : first + chunk);
    }
  }
  // Items of slice s that its waves take without a claim (blocks of one
  // wavefront).
  __device__ uint32_t slice_first(uint32_t s) const {
    return (gridDim.x - s + kQueueSlices - 1) / kQueueSlices * chunk;
  }
  __device__ uint32_t slice_lo(uint32_t s) const {
    return (uint32_t)((uint64_t)count * s / kQueueSlices);
  }
  // n (wave-uniform, n <= lo) lanes take an item each; `rank` (< n) is this
  // lane's place among them.  A lane that gets no item (the queue is
  // drained) gets 0xFFFFFFFF, which is >= count.  Every item below count is
  // handed out exactly once: each slice's counter hands out its items once,
  // and a wave hands out its claims in order.
  __device__ uint32_t take(uint32_t n, uint32_t rank, uint32_t* queue) {
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t item = 0xFFFFFFFFu, given = 0;
    while (given < n && !drained) {
      if (next == end) {
        const uint32_t lo = slice_lo(slice), len = slice_lo(slice + 1) - lo;
        uint32_t b = slice_first(slice);
        if (b < len) {
          uint32_t a = 0;
          if (lane == 0) a = atomicAdd(queue + slice * kQueueStride, chunk);
          b += __builtin_amdgcn_readfirstlane(a);
        }
        if (b < len) {
          next = lo + b;
          end = lo + (len - b < chunk ? len : b + chunk);
        } else {
          // this slice is exhausted: find one with items left, looking from
          // the next slice on (a counter only grows, so an exhausted slice
          // stays so)
          bool left = false;
          if (lane < kQueueSlices) {
            const uint32_t f = slice_first(lane), n = slice_lo(lane + 1) - slice_lo(lane);
            if (f < n)
              left = __hip_atomic_load(queue + lane * kQueueStride, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT) < n - f;
          }
          const uint32_t m = (uint32_t)__builtin_amdgcn_ballot_w64(left);
          if (m == 0) {
            drained = true;
          } else {
            const uint32_t rot = ((m >> slice) | (m << (kQueueSlices - slice))) & 0xFFu;
            slice = (slice + (uint32_t)__builtin_ctz(rot)) % kQueueSlices;
          }
        }
        continue;
      }
      const uint32_t k = n - given < end - next ? n - given : end - next;
      if (rank >= given && rank - given < k) item = next + (rank - given);
      next += k;
      given += k;
    }
    return item;
  }
};

}  // namespace ngia
