// dev_lanes.hip -- one lane per pair, the whole band window in its registers.
//
// The recurrence is that of dev_align.hip; here a lane keeps the W row words
// of its pair's window and the four bit planes of each (5 W registers), and
// derives a word's match mask from the planes as it is used:
//   t = row & M = row & ~(p0 ^ m0) & ~(p1 ^ m1) & ~(p2 ^ m2) & ~(p3 ^ m3)
// with m_e all ones or all zeros by bit e of the character's code: four
// v_bitop3, then the carry add and one more v_bitop3 for
//   row' = (row + t + cin) | (row & ~M) = (row + t + cin) | (row ^ t).
// A code-0 character (an unknown letter, or past the target's end) matches
// nothing and leaves every row as it is: such characters are skipped.  Words
// outside the record have planes 0, which equal no nonzero code.
//
// Bound: VALU issue.  Six instructions per word and character for 64 pairs,
// no memory and no LDS inside a block.  k_align_win<W> needs three, but its
// table of W x 4 KiB of LDS per wavefront leaves a CU two or three wavefronts
// from W = 9 on, and the segmented kernels spend two to three times their
// algorithmic instructions on lookahead and held words outside the band.
// A wavefront takes 64 pairs together and keeps them to the end: taking new
// pairs lane by lane would merge the window from two copies, which does not
// fit the registers, and the pairs of a bin lie in order of target length, so
// the lanes of a wavefront end within a block of each other.
// Measured, log-normal 1M proteins at -i 50, a bin alone: 586,684 pairs of
// 13 words 0.84 ms with k_align_win<13> and 0.41 here, 553,263 of 15 words
// 0.97 and 0.54; the whole alignment phase (6.0M pairs, 3 to 133 words) 11.2
// and 5.4 ms.  A single pair takes 14 ns per word and character, so a bin
// needs tens of thousands of pairs to pay (kLaneFill).
#include <algorithm>

#include "dev_claim.hpp"
#include "dev_common.hpp"
#include "dev_graph.hpp"

namespace ngia {

namespace {

typedef uint32_t Planes __attribute__((ext_vector_type(4)));
typedef Planes PlanesAt __attribute__((aligned(4)));  // in memory: after a record's length word

// The planes of a word outside its record.
__device__ const uint32_t kZeroPlanes[4] = {0u, 0u, 0u, 0u};

__device__ __forceinline__ Planes load_planes(const uint32_t* p) { return *(const PlanesAt*)p; }

// a & ~(b ^ c)
__device__ __forceinline__ uint32_t and_same(uint32_t a, uint32_t b, uint32_t c) {
  return __builtin_amdgcn_bitop3_b32(a, b, c, 0x90);
}
// a | (b ^ c)
__device__ __forceinline__ uint32_t or_diff(uint32_t a, uint32_t b, uint32_t c) {
  return __builtin_amdgcn_bitop3_b32(a, b, c, 0xF6);
}

template <int W>
struct LaneWindow {
  uint32_t row[W];
  Planes pl[W];
};

// One character against the window: m0..m3 spread its code's bits.  Four
// words at a time, the match masks of the next four between the carry adds of
// these: in program order each instruction would wait for the one before it
// (six in a row per word), and a SIMD holds only two to four wavefronts to
// fill the waits.  The empty asm statements keep the order.
template <int W>
__device__ __forceinline__ void lane_char(LaneWindow<W>& s, uint32_t m0, uint32_t m1, uint32_t m2,
                                          uint32_t m3) {
  uint32_t t[4] = {0u, 0u, 0u, 0u};
  auto level = [&](uint32_t (&v)[4], int j0, int l) {
    #pragma unroll
    for (int i = 0; i < 4; i++) {
      if (j0 + i >= W) continue;
      const Planes& pl = s.pl[j0 + i];
      v[i] = l == 0   ? and_same(s.row[j0 + i], pl.x, m0)
             : l == 1 ? and_same(v[i], pl.y, m1)
             : l == 2 ? and_same(v[i], pl.z, m2)
                      : and_same(v[i], pl.w, m3);
    }
  };
  #pragma unroll
  for (int l = 0; l < 4; l++) {
    level(t, 0, l);
    asm volatile("" : "+v"(t[0]), "+v"(t[1]), "+v"(t[2]), "+v"(t[3]));
  }
  uint32_t cin = 0;
  #pragma unroll
  for (int j0 = 0; j0 < W; j0 += 4) {
    uint32_t u[4] = {0u, 0u, 0u, 0u}, sum[4] = {0u, 0u, 0u, 0u};
    #pragma unroll
    for (int i = 0; i < 4; i++) {
      if (j0 + i < W) {
        uint32_t co;
        sum[i] = __builtin_addc(s.row[j0 + i], t[i], cin, &co);
        cin = co;
      }
      level(u, j0 + 4, i);
      if (i > 0 && j0 + i - 1 < W) s.row[j0 + i - 1] = or_diff(sum[i - 1], s.row[j0 + i - 1], t[i - 1]);
      if (j0 + 4 < W)
        asm volatile("" : "+v"(sum[i]), "+v"(u[0]), "+v"(u[1]), "+v"(u[2]), "+v"(u[3]));
    }
    if (j0 + 3 < W) s.row[j0 + 3] = or_diff(sum[3], s.row[j0 + 3], t[3]);
    #pragma unroll
    for (int i = 0; i < 4; i++) t[i] = u[i];
  }
}

// 64 pairs of a bin of W-word windows: lst[first ..], count pairs in the bin.
template <int W>
__device__ __forceinline__ void lanes_chunk(const AlignArgs& A, const uint2* __restrict__ pairs,
                                            const uint32_t* __restrict__ lst, uint32_t first,
                                            uint32_t count, uint32_t* __restrict__ score,
                                            unsigned long long* tally) {
  constexpr uint32_t kPeriod = W <= kWinMax ? (uint32_t)W : 2u;
  uint64_t ran = 0;
  const uint32_t idx = first + threadIdx.x;
  bool active = idx < count;
  // a lane without a pair runs along on the bin's last one
  const uint32_t p = lst[active ? idx : count - 1u];
  const uint2 pr = pairs[p];
  const uint32_t* rr = A.packed + A.word_off[pr.x] + 1;
  const uint32_t* tp = A.packed + A.word_off[pr.y] + 1;
  const uint32_t R = A.lengths[pr.x], T = A.lengths[pr.y];
  const Band bd = band_edges(R, T, A.thr);
  const int32_t a = (int32_t)(bd.lsft / 32), c = (int32_t)((bd.rsft + 31) / 32);
  const int32_t nw = (int32_t)((R + 31) / 32);
  const uint32_t nb = (T + 31) / 32;
  Planes tn = load_planes(tp);  // the target's next block, loaded a block ahead
  LaneWindow<W> s;
  #pragma unroll
  for (int j = 0; j < W; j++) {  // relative word j <-> absolute j - a
    const int32_t w = j - a;
    s.row[j] = 0xFFFFFFFFu;
    s.pl[j] = load_planes(w >= 0 && w < nw ? rr + 4 * w : kZeroPlanes);
  }
  const uint32_t* ep = rr + 4 * c;  // planes of the next word to enter
  int32_t rem = nw - c;             // words still to enter
  uint32_t cb = 0, lcs = 0, tick = 0;
  do {
    const Planes t = tn;
    // the target's next block (its last one again at the end) and the word
    // that enters after this block, to arrive during it
    if (cb + 1 < nb) tp += 4;
    tn = load_planes(tp);
    const Planes e = load_planes(rem > 0 ? ep : kZeroPlanes);
    const uint32_t nz = t.x | t.y | t.z | t.w;  // characters with a nonzero code
    if (__builtin_amdgcn_ballot_w64(active && nz != 0xFFFFFFFFu) == 0) {
      #pragma unroll 1
      for (uint32_t k = 0; k < 32; k++)
        lane_char<W>(s, (uint32_t)__builtin_amdgcn_sbfe((int)t.x, k, 1),
                     (uint32_t)__builtin_amdgcn_sbfe((int)t.y, k, 1),
                     (uint32_t)__builtin_amdgcn_sbfe((int)t.z, k, 1),
                     (uint32_t)__builtin_amdgcn_sbfe((int)t.w, k, 1));
    } else {
      #pragma unroll 1
      for (uint32_t k = 0; k < 32; k++)
        if (active && ((nz >> k) & 1u))
          lane_char<W>(s, (uint32_t)__builtin_amdgcn_sbfe((int)t.x, k, 1),
                       (uint32_t)__builtin_amdgcn_sbfe((int)t.y, k, 1),
                       (uint32_t)__builtin_amdgcn_sbfe((int)t.z, k, 1),
                       (uint32_t)__builtin_amdgcn_sbfe((int)t.w, k, 1));
    }
    // slide: word 0 leaves, the next one enters at the top
    lcs += 32u - __popc(s.row[0]);
    #pragma unroll
    for (int j = 0; j + 1 < W; j++) {
      s.row[j] = s.row[j + 1];
      s.pl[j] = s.pl[j + 1];
    }
    s.row[W - 1] = 0xFFFFFFFFu;
    s.pl[W - 1] = e;
    ep += 4;
    rem--;
    cb++;
    tick++;
    const bool end = cb >= nb;
    if (active && (end || tick == kPeriod)) {
      uint32_t all = lcs;
      #pragma unroll
      for (int j = 0; j < W; j++) all += 32u - __popc(s.row[j]);
      const bool fail = !end && !A.raw_lcs && cannot_pass(all, 32u * cb, R, T, A.thr);
      if (end || fail) {
        score[p] = fail ? 0u : pair_value(A, all, R, T);
        if (tally) ran += ref_tiles(R, T, A.thr, end ? nb : cb);
        active = false;
      }
    }
    if (tick == kPeriod) tick = 0;
  } while (__builtin_amdgcn_ballot_w64(active) != 0);
  if (tally && ran) atomicAdd(tally, (unsigned long long)ran);
}

// A bin's chunks are cut into eight runs, one per XCD (blockIdx.x mod 8 under
// the round-robin dispatch of workgroups), so that neighbouring pairs, which
// share records, meet in one L2.  Chunk `c` of XCD x's runs, counted from the
// class's widest bin down; false past the end, when *c is what is left of it.
template <int LO, int W>
__device__ __forceinline__ bool lanes_at(const AlignArgs& A, const uint2* pairs, const uint32_t* list,
                                         const uint32_t* bin_off, const uint32_t* bin_cnt,
                                         uint32_t* score, unsigned long long* tally, uint32_t wlo,
                                         uint32_t whi, uint32_t x, uint32_t c) {
  constexpr int bin = lane_bin(W);
  const uint32_t count = (uint32_t)W >= wlo && (uint32_t)W <= whi ? bin_cnt[bin] : 0u;
  const uint64_t chunks = (count + 63) / 64;
  const uint32_t lo = (uint32_t)(chunks * x / 8), len = (uint32_t)(chunks * (x + 1) / 8) - lo;
  if (c < len) {
    lanes_chunk<W>(A, pairs, list + bin_off[bin], 64 * (lo + c), count, score,
                   tally ? tally + bin : nullptr);
    return true;
  }
  if constexpr (W > LO)
    return lanes_at<LO, W - 1>(A, pairs, list, bin_off, bin_cnt, score, tally, wlo, whi, x, c - len);
  else
    return false;
}

}  // namespace

// A wavefront's first chunk is the one of its number on its XCD, its others
// come from the XCD's counter and then from those of the other XCDs.  A round
// whose chunks are all somebody's first touches no counter: with every
// wavefront asking every bin's queue, the queues of 45,000 pairs took longer
// than their alignment (0.39 against 0.28 ms for the graph of 10,000
// proteins at -i 70).
template <int LO, int HI, int EU>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(EU, EU))) void k_align_lanes(
    AlignArgs A, const uint2* __restrict__ pairs, const uint32_t* __restrict__ list,
    const uint32_t* __restrict__ bin_off, const uint32_t* __restrict__ bin_cnt,
    uint32_t* __restrict__ next, uint32_t* __restrict__ score, unsigned long long* tally,
    uint32_t wlo, uint32_t whi) {
  for (uint32_t k = 0; k < 8; k++) {
    const uint32_t x = (blockIdx.x + k) % 8;
    uint32_t total = 0;
    for (uint32_t W = wlo; W <= whi; W++) {
      const uint64_t chunks = (bin_cnt[lane_bin((int)W)] + 63) / 64;
      total += (uint32_t)(chunks * (x + 1) / 8) - (uint32_t)(chunks * x / 8);
    }
    const uint32_t waves = (gridDim.x - x + 7) / 8;  // of this XCD
    uint32_t c = blockIdx.x / 8;
    bool first = k == 0;
    for (;;) {
      if (!first) {
        if (waves >= total) break;  // every chunk is some wavefront's first
        uint32_t a = 0;
        if (threadIdx.x == 0) a = atomicAdd(next + x * kQueueStride, 1u);
        c = waves + __builtin_amdgcn_readfirstlane(a);
      }
      first = false;
      if (c >= total) break;
      lanes_at<LO, HI>(A, pairs, list, bin_off, bin_cnt, score, tally, wlo, whi, x, c);
    }
  }
}

// The width classes: bounds of W, and the wavefronts per SIMD that 5 W + 40
// registers allow.  One launch walks a class's bins from the widest down, so
// the tail of one bin is filled by the next.
#define NGIA_LANE_CLASSES(X) X(0, 2, 8, 6) X(1, 9, 16, 4) X(2, 17, 24, 3) X(3, 25, 40, 2)

void launch_align_lanes(int cls, const AlignArgs& a, const uint2* pairs, const uint32_t* list,
                        const uint32_t* bin_off, const uint32_t* bin_cnt, uint32_t* queue,
                        uint32_t* score, unsigned long long* tally, uint32_t wlo, uint32_t whi,
                        uint32_t cus, uint64_t max_pairs, hipStream_t stream) {
  if (!a.lengths) throw HipError{NGIA_ERR_ARG, "binned alignment without record lengths"};
  // a chunk per 64 pairs and one more per bin, cut into runs for eight XCDs
  const uint64_t need = (max_pairs + 63) / 64 + (whi - wlo + 1) + 64;
  uint32_t* next = queue + (size_t)lane_bin((int)whi) * kQueueWords;
  switch (cls) {
#define X(C, LO, HI, EU)                                                                          \
  case C:                                                                                         \
    hipLaunchKernelGGL((k_align_lanes<LO, HI, EU>),                                               \
                       dim3((uint32_t)std::min<uint64_t>(need, (uint64_t)cus * 4 * EU)), dim3(64), \
                       0, stream, a, pairs, list, bin_off, bin_cnt, next, score, tally, wlo, whi); \
    break;
    NGIA_LANE_CLASSES(X)
#undef X
    default:
      throw HipError{NGIA_ERR_ARG, "no such width class"};
  }
  NGIA_HIP(hipGetLastError());
}

}  // namespace ngia
