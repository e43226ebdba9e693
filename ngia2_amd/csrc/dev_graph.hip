// dev_graph.hip -- candidate pairs, pair binning and edge emission for the
// graph build (buildGraph.hpp:256-363) and fast mode (fastClustering.hpp:249-352).
//
// Every kernel here has a grid that depends only on host-known sizes (n,
// bands, a persistent grid) and reads data-dependent counts from device
// memory, so a whole round can be captured in a hipGraph.  Counters are
// cleared with a fill kernel, never with hipMemsetAsync.
#include <algorithm>
#include <cstring>

#include <rocprim/rocprim.hpp>

#include "dev_common.hpp"
#include "dev_graph.hpp"

namespace ngia {

__global__ void k_fill_u32(uint32_t* __restrict__ p, uint32_t v, uint64_t count) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count;
       i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

void fill_u32(uint32_t* p, uint32_t v, uint64_t count, hipStream_t s) {
  if (count == 0) return;
  uint64_t blocks = (count + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)blocks), dim3(256), 0, s, p, v, count);
  NGIA_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ scan
// Exclusive scan of n uint32 into n+1 uint64 (out[n] = total), both at 16-byte
// aligned addresses, over tiles of 4,096.  A tile's block adds up what lies
// before it: the sums of the tiles (k_scan_reduce), or, up to kScanDirect
// elements, the elements themselves, in one launch.  With a pass of its own for
// the tiles' prefix, by a single block, 10,000 elements took 17 us in three
// launches and 1 million 23; so 5 in one and 14 in two.
constexpr uint32_t kScanTile = 4096;
constexpr uint32_t kScanDirect = 4 * kScanTile;

__device__ inline uint64_t wave_sum(uint64_t x) {
  #pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
  return x;
}

__global__ __launch_bounds__(256) void k_scan_reduce(const uint32_t* __restrict__ in, uint32_t n,
                                                     uint64_t* __restrict__ sums) {
  __shared__ uint64_t red[4];
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile;
  uint64_t s = 0;
  #pragma unroll
  for (uint32_t k = 0; k < kScanTile / 256; k++) {
    const uint64_t i = base + 256 * k + threadIdx.x;
    if (i < n) s += in[i];
  }
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) sums[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

__global__ __launch_bounds__(256) void k_scan_apply(const uint32_t* __restrict__ in, uint32_t n,
                                                    const uint64_t* __restrict__ sums,
                                                    uint64_t* __restrict__ out) {
  __shared__ uint64_t red[4], sh[4];
  const uint32_t t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile;
  // each thread owns 16 consecutive elements
  const uint64_t mine = base + (uint64_t)t * 16;
  uint32_t v[16];
  const bool full = mine + 16 <= n;
  if (full) {
    #pragma unroll
    for (int k = 0; k < 4; k++) {
      const uint4 q = ((const uint4*)(in + mine))[k];
      v[4 * k] = q.x;
      v[4 * k + 1] = q.y;
      v[4 * k + 2] = q.z;
      v[4 * k + 3] = q.w;
    }
  } else {
    #pragma unroll
    for (int k = 0; k < 16; k++) {
      const uint32_t q = n ? in[mine + k < n ? mine + k : n - 1] : 0u;
      v[k] = mine + k < n ? q : 0u;
    }
  }
  uint64_t before = 0;
  if (sums) {
    for (uint32_t k = t; k < blockIdx.x; k += 256) before += sums[k];
  } else {  // every load before the first sum: each waits for another XCD's write
    uint32_t b[kScanDirect / kScanTile - 1][kScanTile / 256];
    #pragma unroll
    for (uint32_t tile = 0; tile < kScanDirect / kScanTile - 1; tile++)
      #pragma unroll
      for (uint32_t k = 0; k < kScanTile / 256; k++)
        b[tile][k] = tile < blockIdx.x ? in[tile * kScanTile + 256 * k + t] : 0u;
    #pragma unroll
    for (uint32_t tile = 0; tile < kScanDirect / kScanTile - 1; tile++)
      #pragma unroll
      for (uint32_t k = 0; k < kScanTile / 256; k++) before += b[tile][k];
  }
  before = wave_sum(before);
  uint64_t s = 0;
  #pragma unroll
  for (int k = 0; k < 16; k++) s += v[k];
  uint64_t x = s;  // inclusive prefix over the wavefront
  #pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint64_t y = __shfl_up(x, o);
    if (lane >= (uint32_t)o) x += y;
  }
  if (lane == 0) red[wave] = before;
  if (lane == 63) sh[wave] = x;
  __syncthreads();
  uint64_t run = red[0] + red[1] + red[2] + red[3] + x - s;
  for (uint32_t w = 0; w < wave; w++) run += sh[w];
  uint64_t o[16];
  #pragma unroll
  for (int k = 0; k < 16; k++) {
    o[k] = run;
    run += v[k];
  }
  if (full) {
    #pragma unroll
    for (int k = 0; k < 8; k++)
      ((ulonglong2*)(out + mine))[k] = make_ulonglong2(o[2 * k], o[2 * k + 1]);
  } else {
    #pragma unroll
    for (int k = 0; k < 16; k++)
      if (mine + k < n) out[mine + k] = o[k];
  }
  if (blockIdx.x == gridDim.x - 1 && t == 255) out[n] = run;
}

uint64_t scan_scratch_words(uint32_t n) { return (n + kScanTile - 1) / kScanTile + 2; }

void scan_u32(const uint32_t* in, uint32_t n, uint64_t* out, uint64_t* sums, hipStream_t s) {
  const uint32_t nb = n ? (n + kScanTile - 1) / kScanTile : 1u;
  const bool direct = n <= kScanDirect;
  if (!direct) hipLaunchKernelGGL(k_scan_reduce, dim3(nb), dim3(256), 0, s, in, n, sums);
  hipLaunchKernelGGL(k_scan_apply, dim3(nb), dim3(256), 0, s, in, n,
                     direct ? (const uint64_t*)nullptr : sums, out);
  NGIA_HIP(hipGetLastError());
}

// ------------------------------------------------------------- predicate
// Candidate predicate of buildGraph.hpp:262-266: rep[i] != i and
// (float)len[i] >= (float)len[rep[i]] * thr.
__device__ inline bool is_job(uint32_t r, uint32_t i, const uint32_t* len, float thr) {
  return r != i && (float)len[i] >= (float)len[r] * thr;
}

// ------------------------------------------------------------- plain form
// Per band: flags, scan, then job triplets in ascending i (buildGraph.hpp:278-321).
__global__ void k_band_flags(const uint32_t* __restrict__ rep, const uint32_t* __restrict__ len,
                             uint32_t n, float thr, const uint32_t* __restrict__ parent,
                             uint32_t* __restrict__ flags) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t r = rep[i];
  // fast mode (fastClustering.hpp:256-258) has no length filter, only "unclustered"
  flags[i] = parent ? (uint32_t)(r != i && parent[i] == 0xFFFFFFFFu) : (uint32_t)is_job(r, i, len, thr);
}

__global__ void k_band_jobs(const uint32_t* __restrict__ rep, const uint32_t* __restrict__ flags,
                            const uint64_t* __restrict__ pos, uint32_t n,
                            uint32_t* __restrict__ jobs) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || !flags[i]) return;
  const uint64_t j = pos[i];
  jobs[3 * j] = rep[i];
  jobs[3 * j + 1] = i;
  jobs[3 * j + 2] = 0;
}

void band_jobs(const uint32_t* rep, const uint32_t* len, uint32_t n, float thr,
               const uint32_t* parent, uint32_t* flags, uint64_t* pos, uint64_t* sums,
               uint32_t* jobs, hipStream_t s) {
  hipLaunchKernelGGL(k_band_flags, dim3(grid_for(n, 256)), dim3(256), 0, s, rep, len, n, thr,
                     parent, flags);
  NGIA_HIP(hipGetLastError());
  scan_u32(flags, n, pos, sums, s);
  hipLaunchKernelGGL(k_band_jobs, dim3(grid_for(n, 256)), dim3(256), 0, s, rep, flags, pos, n, jobs);
  NGIA_HIP(hipGetLastError());
}

// Slot of this lane in an append-only list: one atomic per wavefront for the
// lanes with `pred` set; returns ~0ull for lanes without it.
__device__ inline unsigned long long wave_append(unsigned long long* counter, bool pred) {
  const uint64_t m = __builtin_amdgcn_ballot_w64(pred);
  if (!m) return ~0ull;
  const uint32_t lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  const uint32_t leader = (uint32_t)__builtin_ctzll(m);
  unsigned long long base = 0;
  if (lane == leader) base = atomicAdd(counter, (unsigned long long)__builtin_popcountll(m));
  base = __shfl(base, (int)leader);
  const uint32_t rank = (uint32_t)__builtin_popcountll(m & ((1ull << lane) - 1ull));
  return pred ? base + rank : ~0ull;
}

// Append the passing jobs of one band to the raw edge list.
__global__ void k_jobs_to_edges(const uint32_t* __restrict__ jobs, uint32_t count,
                                uint64_t* __restrict__ ekeys, uint32_t* __restrict__ escores,
                                unsigned long long* __restrict__ ecount) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t sc = j < count ? jobs[3 * j + 2] : 0u;
  const unsigned long long at = wave_append(ecount, sc != 0);
  if (sc == 0) return;
  ekeys[at] = ((uint64_t)jobs[3 * j] << 32) | jobs[3 * j + 1];
  escores[at] = sc;
}

void jobs_to_edges(const uint32_t* jobs, uint32_t count, uint64_t* ekeys, uint32_t* escores,
                   unsigned long long* ecount, hipStream_t s) {
  if (count == 0) return;
  hipLaunchKernelGGL(k_jobs_to_edges, dim3(grid_for(count, 256)), dim3(256), 0, s, jobs, count,
                     ekeys, escores, ecount);
  NGIA_HIP(hipGetLastError());
}

// Fast mode: parent[tar] = rep for each passing job of the band.
__global__ void k_fast_apply(const uint32_t* __restrict__ jobs, uint32_t count,
                             uint32_t* __restrict__ parent) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= count) return;
  if (jobs[3 * j + 2] > 0) parent[jobs[3 * j + 1]] = jobs[3 * j];
}

void fast_apply(const uint32_t* jobs, uint32_t count, uint32_t* parent, hipStream_t s) {
  if (count == 0) return;
  hipLaunchKernelGGL(k_fast_apply, dim3(grid_for(count, 256)), dim3(256), 0, s, jobs, count,
                     parent);
  NGIA_HIP(hipGetLastError());
}

// One thread per target that has no parent yet: its kept pairs of the round in
// band order; the first that passes gives its parent.  The reference aligns the
// target in every band up to that one (in all of them when none passes):
// *total counts those bands.
__global__ __launch_bounds__(256) void k_fast_resolve(uint32_t n, const uint64_t* __restrict__ off,
                                                      const uint2* __restrict__ pairs,
                                                      const uint32_t* __restrict__ score,
                                                      const uint64_t* __restrict__ keep,
                                                      FastRound fast,
                                                      unsigned long long* __restrict__ total) {
  __shared__ unsigned long long sum;
  if (threadIdx.x == 0) sum = 0;
  __syncthreads();
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  uint32_t aligned = 0;
  if (i < n && fast.parent[i] == 0xFFFFFFFFu) {
    uint64_t left = keep[i];
    const uint64_t valid = fast.valid[i];
    bool pass = false;
    for (uint64_t p = off[i]; left; p++, left &= left - 1) {
      if (!score[p]) continue;
      fast.parent[i] = pairs[p].x;
      const uint32_t b = (uint32_t)__builtin_ctzll(left);
      aligned = (uint32_t)__builtin_popcountll(valid & ((2ull << b) - 1ull));
      pass = true;
      break;
    }
    if (!pass && fast.last) aligned = (uint32_t)__builtin_popcountll(valid);
  }
  if (aligned) atomicAdd(&sum, (unsigned long long)aligned);
  __syncthreads();
  if (threadIdx.x == 0 && sum) atomicAdd(total, sum);
}

void fast_resolve(uint32_t n, const uint64_t* off, const uint2* pairs, const uint32_t* score,
                  const uint64_t* keep, const FastRound& fast, unsigned long long* total,
                  hipStream_t s) {
  hipLaunchKernelGGL(k_fast_resolve, dim3(grid_for(n, 256)), dim3(256), 0, s, n, off, pairs, score,
                     keep, fast, total);
  NGIA_HIP(hipGetLastError());
}

// ------------------------------------------------------------- batched form
// Count pass: a block takes 64 consecutive targets.  The 64 x 64 tile
// rep[b][i0..i0+63] is read row by row (coalesced) into LDS; each wavefront
// handles 16 targets, lane b holding rep[b][i].  The lengths of all 16
// targets and their representatives are gathered before the first is tested,
// so the wave waits on memory once, not 16 times.  The distinct
// representatives passing the candidate predicate are kept in order of their
// first band: keep[i] has bit b set for the band that contributes each kept
// representative, cnt[i] = its popcount, and *total gains the candidate
// count with duplicates.
__device__ inline void load_rep_tile(const uint32_t* __restrict__ rep, uint32_t n, uint32_t bands,
                                     uint32_t i0, uint32_t (&tile)[64][65]) {
  // all 16 loads of a thread before the first store (unconditional, index 0 where
  // there is nothing to load): one at a time they took 16 us of a small round
  const uint32_t t = threadIdx.x & 63u, b0 = threadIdx.x >> 6;
  uint32_t v[16];
  #pragma unroll
  for (uint32_t k = 0; k < 16; k++) {
    const uint32_t b = b0 + 4 * k;
    v[k] = rep[b < bands && i0 + t < n ? (uint64_t)b * n + i0 + t : 0u];
  }
  #pragma unroll
  for (uint32_t k = 0; k < 16; k++) tile[b0 + 4 * k][t] = v[k];
}

__global__ __launch_bounds__(256) void k_pair_count(const uint32_t* __restrict__ rep,
                                                    const uint32_t* __restrict__ len, uint32_t n,
                                                    uint32_t t0, uint32_t bands, float thr,
                                                    FastRound fast, uint32_t* __restrict__ cnt,
                                                    uint64_t* __restrict__ keep_out,
                                                    uint32_t* __restrict__ degree,
                                                    unsigned long long* __restrict__ total) {
  __shared__ uint32_t tile[64][65];
  __shared__ unsigned long long btotal;
  const uint32_t i0 = blockIdx.x * 64;
  if (degree && threadIdx.x < 64 && i0 + threadIdx.x < n) degree[i0 + threadIdx.x] = 0;
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (threadIdx.x == 0) btotal = 0;
  load_rep_tile(rep, n, bands, i0, tile);
  __syncthreads();
  uint32_t lr[16], li[16];
  uint32_t need = 0;  // bit tt: lane's band has a representative other than the target
  #pragma unroll
  for (int tt = 0; tt < 16; tt++) {
    const uint32_t t = wave * 16 + tt, i = i0 + t;
    const uint32_t r = tile[lane][t];
    const bool nd = lane < bands && i < n && i >= t0 && r != i;
    lr[tt] = len[nd ? r : 0u];  // unconditional: rows hold indices < n
    li[tt] = len[i < n ? i : 0u];
    need |= (uint32_t)nd << tt;
  }
  uint32_t wtotal = 0;
  #pragma unroll
  for (int tt = 0; tt < 16; tt++) {
    const uint32_t t = wave * 16 + tt;
    const uint32_t i = i0 + t;
    if (i >= n) break;
    const uint32_t r = tile[lane][t];
    // is_job: r != i and (float)len[i] >= (float)len[r] * thr; the fast mode has
    // no length test (fastClustering.hpp:256-258)
    const bool valid =
        ((need >> tt) & 1u) && (fast.parent || (float)li[tt] >= (float)lr[tt] * thr);
    const uint64_t vm = __builtin_amdgcn_ballot_w64(valid);
    uint64_t mask = vm, keep = 0;
    while (mask) {
      const uint32_t b0 = (uint32_t)__builtin_ctzll(mask);
      const uint32_t r0 = __builtin_amdgcn_readlane(r, b0);
      keep |= 1ull << b0;
      mask &= ~__builtin_amdgcn_ballot_w64(valid && r == r0);
    }
    if (fast.parent) {
      keep = fast.parent[i] == 0xFFFFFFFFu ? keep & fast.bands : 0ull;
      if (lane == 0) fast.valid[i] = vm;
    }
    if (lane == 0) {
      cnt[i] = (uint32_t)__builtin_popcountll(keep);
      keep_out[i] = keep;
    }
    wtotal += (uint32_t)__builtin_popcountll(vm);
  }
  if (lane == 0 && wtotal) atomicAdd(&btotal, (unsigned long long)wtotal);
  __syncthreads();
  if (threadIdx.x == 0 && btotal) atomicAdd(total, btotal);
}

// Emit pass: the same tile; target i's kept representatives, in band order,
// go to pairs[off[i] ..].
__global__ __launch_bounds__(256) void k_pair_emit(const uint32_t* __restrict__ rep, uint32_t n,
                                                   uint32_t bands,
                                                   const uint64_t* __restrict__ keep_in,
                                                   const uint64_t* __restrict__ off,
                                                   uint2* __restrict__ pairs) {
  __shared__ uint32_t tile[64][65];
  const uint32_t i0 = blockIdx.x * 64;
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // lane tt of a wavefront: target tt's kept bands and first pair, loaded once (a
  // load of both for each of the 16 targets: 104 us at 1M records, so 52)
  const uint32_t mine = i0 + wave * 16 + (lane & 15u);
  const uint64_t kept = keep_in[mine < n ? mine : n - 1], first = off[mine < n ? mine : n - 1];
  load_rep_tile(rep, n, bands, i0, tile);
  __syncthreads();
  #pragma unroll
  for (int tt = 0; tt < 16; tt++) {
    const uint32_t t = wave * 16 + tt;
    const uint32_t i = i0 + t;
    if (i >= n) break;
    auto of_target = [&](uint64_t x) {
      const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)x, tt);
      const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(x >> 32), tt);
      return ((uint64_t)hi << 32) | lo;
    };
    const uint64_t keep = of_target(kept), at = of_target(first);
    if ((keep >> lane) & 1ull) {
      const uint32_t rank = (uint32_t)__builtin_popcountll(keep & ((1ull << lane) - 1ull));
      pairs[at + rank] = make_uint2(tile[lane][t], i);
    }
  }
}

void pair_count(const uint32_t* rep, const uint32_t* len, uint32_t n, uint32_t t0, uint32_t bands,
                float thr, uint32_t* cnt, uint64_t* keep, uint32_t* degree,
                unsigned long long* total, hipStream_t s, const FastRound& fast) {
  hipLaunchKernelGGL(k_pair_count, dim3((n + 63) / 64), dim3(256), 0, s, rep, len, n, t0, bands,
                     thr, fast, cnt, keep, degree, total);
  NGIA_HIP(hipGetLastError());
}

void pair_emit(const uint32_t* rep, uint32_t n, uint32_t bands, const uint64_t* keep,
               const uint64_t* off, uint2* pairs, hipStream_t s) {
  hipLaunchKernelGGL(k_pair_emit, dim3((n + 63) / 64), dim3(256), 0, s, rep, n, bands, keep, off,
                     pairs);
  NGIA_HIP(hipGetLastError());
}

// Bin of a pair by its band window: W = a + c words.  A bin per width up to
// kLaneMax words, which k_bin_offsets routes to the shape that aligns it; two
// bins of the segmented kernels up to 60 words;
// larger windows to k_align_wave<K> with the smallest K in {1,2,4,...,32}
// with 64K >= W + K - 1 (the wave trails the band bottom in steps of K
// words); T == 0 scores 0 at once (its LCS is 0, so the pass test fails);
// anything wider goes to the plain kernel.
__device__ inline uint32_t pair_bin(uint32_t R, uint32_t T, float thr, uint32_t kmax,
                                    uint64_t* tiles) {
  if (length_rejects(R, T, thr) || T == 0) {
    *tiles = 0;
    return kBinZero;
  }
  const Band bd = band_edges(R, T, thr);
  const uint32_t a = bd.lsft / 32, c = (bd.rsft + 31) / 32, W = a + c;
  *tiles = ref_tiles(R, T, thr, (T + 31) / 32);
  if (W <= (uint32_t)kWinMax) return W;  // W >= 2 whenever T > 0
  if (W <= (uint32_t)kLaneMax) return (uint32_t)lane_bin((int)W);
  if (W <= 45) return kBinSeg16x3;
  if (W <= 60) return kBinSeg16x4;
  for (uint32_t k = 0, K = 1; K <= kmax; k++, K <<= 1)
    if (W + K - 1 <= 64u * (uint32_t)K) return kBinWave0 + k;
  return kBinPlain;
}

__global__ void k_bin_count(const uint2* __restrict__ pairs, const uint64_t* __restrict__ npairs,
                            const uint32_t* __restrict__ len, float thr, uint32_t kmax,
                            uint32_t* __restrict__ bin_of, uint32_t* __restrict__ bin_cnt,
                            unsigned long long* __restrict__ bin_tiles,
                            uint32_t* __restrict__ score) {
  const uint64_t P = *npairs;
  __shared__ uint32_t local[kBins];
  __shared__ unsigned long long ltiles[kBins];
  if (threadIdx.x < kBins) {
    local[threadIdx.x] = 0;
    ltiles[threadIdx.x] = 0;
  }
  __syncthreads();
  for (uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; p < P;
       p += (uint64_t)gridDim.x * blockDim.x) {
    const uint2 pr = pairs[p];
    uint64_t t;
    const uint32_t b = pair_bin(len[pr.x], len[pr.y], thr, kmax, &t);
    bin_of[p] = b;
    if (b == kBinZero) score[p] = 0;
    atomicAdd(&local[b], 1u);
    if (t) atomicAdd(&ltiles[b], (unsigned long long)t);
  }
  __syncthreads();
  if (threadIdx.x < kBins && local[threadIdx.x]) {
    atomicAdd(&bin_cnt[threadIdx.x], local[threadIdx.x]);
    atomicAdd(&bin_tiles[threadIdx.x], ltiles[threadIdx.x]);
  }
}

// Route window bins by the tuned shapes (remap[b] = the bin that aligns bin
// b's pairs, counts and tiles moved along), then bin_off[b] = exclusive prefix
// of bin_cnt; also resets the scatter cursors.  One thread routes, over
// copies in LDS: a chain of dependent global accesses took longer than the
// counting.
__global__ __launch_bounds__(64) void k_bin_offsets(uint32_t* __restrict__ bin_cnt,
                                                    uint32_t* __restrict__ bin_off,
                                                    uint32_t* __restrict__ cursor,
                                                    uint32_t* __restrict__ remap,
                                                    unsigned long long* __restrict__ bin_tiles,
                                                    RouteTable route, uint32_t seg2_min,
                                                    uint32_t lane_fill, bool compact,
                                                    uint32_t* __restrict__ host_cnt) {
  __shared__ uint32_t cnt[kBins], to_bin[kBins], off[64];
  __shared__ unsigned long long tiles[kBins];
  static_assert(kBins < 64, "one thread per bin, and one for the end");
  const uint32_t t = threadIdx.x;
  if (t < (uint32_t)kBins) {
    cnt[t] = bin_cnt[t];
    tiles[t] = bin_tiles[t];
    to_bin[t] = t;
    cursor[t] = 0;
  }
  const bool lanes_off = lane_fill == 0xFFFFFFFFu;
  // the tiles of the bins that a lane per pair could take past kWinLds words
  const int width = t < (uint32_t)kBins ? bin_width((int)t) : 0;
  const uint64_t total = wave_sum(width > kWinLds ? bin_tiles[t] : 0ull);
  if (route.class_size[0] == 0 && !compact && lane_fill != 0 && !lanes_off) {
    // Few pairs in all: a wavefront each (kWaveAllPairs).
    const uint32_t c = t > 0 && t < (uint32_t)kBins ? bin_cnt[t] : 0u;
    const bool narrow = width > kWaveAllMin || is_seg_bin((int)t);
    const uint64_t wider = __builtin_amdgcn_ballot_w64(c != 0 && width < 2 && !narrow);
    const uint64_t all = wider ? ~0ull : wave_sum(c);
    if (all <= kWaveAllPairs) {
      const uint64_t n1 = wave_sum(narrow ? c : 0u), t1 = wave_sum(narrow && c ? bin_tiles[t] : 0ull);
      if (narrow && c) {
        to_bin[t] = (uint32_t)kBinWave0;
        cnt[t] = 0;
        tiles[t] = 0;
      }
      if (t == (uint32_t)kBinWave0) {
        cnt[t] += (uint32_t)n1;
        tiles[t] += t1;
      }
    }
  }
  __syncthreads();
  if (t == 0) {
    auto move = [&](int from, int to) {
      if (!cnt[from] || from == to) return;
      to_bin[from] = (uint32_t)to;
      cnt[to] += cnt[from];
      tiles[to] += tiles[from];
      cnt[from] = 0;
      tiles[from] = 0;
    };
    const bool tuned = route.class_size[0] != 0;
    // Whether one lane per pair pays for `c` pairs of `t` tiles in all.
    auto lanes_pay = [&](uint32_t c, unsigned long long t) {
      const unsigned long long few = (unsigned long long)kLaneTiles * c;
      return !lanes_off && (t <= few || total * c >= (unsigned long long)lane_fill * (t - few));
    };
    // Window bins: the tuned shape; without a table, kWinLds+1..kWinMax words
    // by lanes_pay, and where it does not pay a wavefront or a segment per
    // pair.  Compact alphabets have their own window kernels.
    uint32_t small = 0;
    for (int W = 2; W <= kWinMax; W++) {
      if (!cnt[W]) continue;
      if (tuned) {
        move(W, (int)route_window_bin(route, (uint32_t)W, cnt[W]));
      } else if (!compact && !lanes_off && W > kWinLds && !lanes_pay(cnt[W], tiles[W])) {
        small += cnt[W];
      }
      if (!compact && W <= kWinLds && cnt[W] < kLowLanePairs) move(W, lane_bin(W));
    }
    if (small)
      for (int W = kWinLds + 1; W <= kWinMax; W++)
        if (cnt[W] && !lanes_pay(cnt[W], tiles[W]))
          move(W, small <= kWavePairs ? kBinWave0 : W <= 14 ? kBinSeg8x2 : kBinSeg32);
    // Windows of 17-60 words in four groups (and W = 31 by itself).  Up to
    // kLaneMax words a group may keep one lane per pair, a bin per width.
    // Else: several words per lane (four or eight pairs per wavefront) when
    // the group has the pairs to fill the device that way; a smaller one
    // (long pairs, every segment in flight at once either way) one word per
    // lane, whose per-character chain is shorter, or a wavefront per pair.
    // The tuned table decides by the group's size class, or leaves it to
    // lanes_pay and the size limit seg2_min (NGIA_LONG_DEFAULT).
    auto group = [&](int w0, int w1, int extra, int multi, int single, int g) {
      uint32_t n2 = extra >= 0 ? cnt[extra] : 0u, nl = 0;
      unsigned long long tl = 0;
      for (int W = w0; W <= w1; W++) {
        nl += cnt[lane_bin(W)];
        tl += tiles[lane_bin(W)];
      }
      n2 += nl;
      if (!n2) return;
      const uint32_t choice =
          g < 0 || !tuned ? NGIA_LONG_DEFAULT : route.lng[g][route_class(route, n2)];
      const bool lanes = choice == NGIA_LONG_MULTI ? !lanes_off && n2 >= kLaneMinPairs
                                                   : choice == NGIA_LONG_DEFAULT && lanes_pay(nl, tl);
      const bool several = choice == NGIA_LONG_MULTI ||
                           (choice == NGIA_LONG_DEFAULT && n2 >= seg2_min);
      const int to = several ? multi : single;
      if (!lanes)
        for (int W = w0; W <= w1; W++) move(lane_bin(W), to);
      if (extra >= 0) move(extra, to);  // the windows too wide for a lane
    };
    group(17, 21, -1, kBinSeg8x3, kBinSeg32, 0);
    group(22, 30, -1, kBinSeg16x2, kBinSeg32, 1);
    group(31, 31, -1, kBinSeg32, kBinSeg32, -1);
    group(32, kLaneMax, kBinSeg16x3, kBinSeg16x3, kBinWave0, 2);
    group(1, 0, kBinSeg16x4, kBinSeg16x4, kBinWave0, 3);
  }
  __syncthreads();
  const uint32_t c = t < (uint32_t)kBins ? cnt[t] : 0u;
  uint32_t x = c;
  #pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, o);
    if (t >= (uint32_t)o) x += y;
  }
  off[t] = x - c;
  if (t < (uint32_t)kBins) {
    bin_cnt[t] = cnt[t];
    if (host_cnt) host_cnt[t] = cnt[t];
    bin_tiles[t] = tiles[t];
    remap[t] = to_bin[t];
    bin_off[t] = off[t];
  }
  if (t == (uint32_t)kBins) bin_off[t] = off[t];
}

uint64_t reachable_bins(uint32_t wlo, uint32_t whi, uint64_t pairs, uint32_t kmax,
                        const RouteTable& route, uint32_t lane_fill) {
  uint64_t m = 0;
  auto add = [&](int b) { m |= 1ull << b; };
  const bool each = !route.class_size[0] && lane_fill != 0 && lane_fill != 0xFFFFFFFFu &&
                    pairs <= kWaveAllPairs && whi <= 60;  // a wavefront per pair
  if (each && whi >= 2) add(kBinWave0);
  for (uint32_t W = std::max(wlo, 2u); each && W <= std::min(whi, (uint32_t)kWaveAllMin); W++)
    add(lane_bin((int)W));
  for (uint32_t W = std::max(wlo, 2u); !each && W <= std::min(whi, 60u); W++) {
    add(kBinWave0);
    if (W <= (uint32_t)kWinMax) {
      if (W > (uint32_t)kWinLds || pairs >= kLowLanePairs) add((int)W);
      add(lane_bin((int)W));
      add(kBinSeg8x2);
      add(kBinSeg32);
      if (route.class_size[0]) add(kBinSeg16);
    } else if (W <= 31) {
      add(lane_bin((int)W));
      add(W <= 21 ? kBinSeg8x3 : kBinSeg16x2);
      add(kBinSeg32);
    } else {
      if (W <= (uint32_t)kLaneMax) add(lane_bin((int)W));
      add(W <= 45 ? kBinSeg16x3 : kBinSeg16x4);
    }
  }
  uint32_t from = 61;  // the narrowest window of the next bin
  for (uint32_t k = 0, K = 1; K <= kmax; k++, K <<= 1) {
    if (whi >= from && wlo <= 64 * K - K + 1) add(kBinWave0 + (int)k);
    from = 64 * K - K + 2;
  }
  if (whi >= from) add(kBinPlain);
  return m;
}

// Scatter pair indices into their bin's segment.  A block takes tiles of
// 4096 pairs: slots are counted in LDS, reserved with one global atomic per
// (tile, bin), then written.
__global__ __launch_bounds__(256) void k_bin_scatter(const uint64_t* __restrict__ npairs,
                                                     const uint32_t* __restrict__ bin_of,
                                                     const uint32_t* __restrict__ remap,
                                                     const uint32_t* __restrict__ bin_off,
                                                     uint32_t* __restrict__ cursor,
                                                     uint32_t* __restrict__ list) {
  __shared__ uint32_t lcnt[kBins], lbase[kBins];
  const uint64_t P = *npairs;
  for (uint64_t base = (uint64_t)blockIdx.x * 4096; base < P; base += (uint64_t)gridDim.x * 4096) {
    if (threadIdx.x < kBins) lcnt[threadIdx.x] = 0;
    __syncthreads();
    uint32_t b[16], pos[16];
    #pragma unroll
    for (int k = 0; k < 16; k++) {
      const uint64_t p = base + (uint64_t)k * 256 + threadIdx.x;
      b[k] = p < P ? remap[bin_of[p]] : 0u;
      pos[k] = p < P ? atomicAdd(&lcnt[b[k]], 1u) : 0u;
    }
    __syncthreads();
    if (threadIdx.x < kBins)
      lbase[threadIdx.x] = lcnt[threadIdx.x] ? atomicAdd(&cursor[threadIdx.x], lcnt[threadIdx.x]) : 0u;
    __syncthreads();
    #pragma unroll
    for (int k = 0; k < 16; k++) {
      const uint64_t p = base + (uint64_t)k * 256 + threadIdx.x;
      if (p < P) list[bin_off[b[k]] + lbase[b[k]] + pos[k]] = (uint32_t)p;
    }
    __syncthreads();
  }
}

void bin_pairs(const uint2* pairs, const uint64_t* npairs, const uint32_t* len, float thr,
               uint32_t* bin_of, uint32_t* bin_cnt, uint32_t* bin_off, uint32_t* cursor,
               uint32_t* list, unsigned long long* bin_tiles, uint32_t* score, uint32_t kmax,
               uint32_t* remap, const RouteTable& route, uint32_t seg2_min, uint32_t lane_fill,
               bool compact, uint32_t grid, hipStream_t s, uint32_t* host_cnt) {
  // A sixteenth of the grid: every block ends with one global atomic per
  // nonempty bin, and a few bins take nearly all pairs, so those counters
  // see one atomic per block.
  hipLaunchKernelGGL(k_bin_count, dim3(std::max(grid / 16, 1u)), dim3(256), 0, s, pairs, npairs, len,
                     thr, kmax, bin_of, bin_cnt, bin_tiles, score);
  hipLaunchKernelGGL(k_bin_offsets, dim3(1), dim3(64), 0, s, bin_cnt, bin_off, cursor, remap,
                     bin_tiles, route, seg2_min, lane_fill, compact, host_cnt);
  hipLaunchKernelGGL(k_bin_scatter, dim3(grid), dim3(256), 0, s, npairs, bin_of, remap, bin_off,
                     cursor, list);
  NGIA_HIP(hipGetLastError());
}

// Job triplets as pairs, and the scores back.
__global__ __launch_bounds__(256) void k_jobs_to_pairs(const uint32_t* __restrict__ jobs, uint32_t count,
                                                       uint2* __restrict__ pairs,
                                                       unsigned long long* __restrict__ npairs) {
  const uint32_t j = blockIdx.x * 256 + threadIdx.x;
  if (j == 0) *npairs = count;
  if (j < count) pairs[j] = make_uint2(jobs[3ull * j], jobs[3ull * j + 1]);
}
__global__ __launch_bounds__(256) void k_scores_to_jobs(const uint32_t* __restrict__ score,
                                                        uint32_t count, uint32_t* __restrict__ jobs) {
  const uint32_t j = blockIdx.x * 256 + threadIdx.x;
  if (j < count) jobs[3ull * j + 2] = score[j];
}
void jobs_to_pairs(const uint32_t* jobs, uint32_t count, uint2* pairs, unsigned long long* npairs,
                   hipStream_t s) {
  hipLaunchKernelGGL(k_jobs_to_pairs, dim3(grid_for(count, 256)), dim3(256), 0, s, jobs, count, pairs,
                     npairs);
  NGIA_HIP(hipGetLastError());
}
void scores_to_jobs(const uint32_t* score, uint32_t count, uint32_t* jobs, hipStream_t s) {
  hipLaunchKernelGGL(k_scores_to_jobs, dim3(grid_for(count, 256)), dim3(256), 0, s, score, count, jobs);
  NGIA_HIP(hipGetLastError());
}

// Pairs of the plain-kernel bin as job triplets, scores copied back after.
__global__ void k_bin_to_jobs(const uint2* __restrict__ pairs, const uint32_t* __restrict__ list,
                              const uint32_t* __restrict__ bin_off, const uint32_t* __restrict__ bin_cnt,
                              uint32_t* __restrict__ jobs) {
  const uint32_t cnt = bin_cnt[kBinPlain], off = bin_off[kBinPlain];
  for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < cnt; j += gridDim.x * blockDim.x) {
    const uint2 pr = pairs[list[off + j]];
    jobs[3 * j] = pr.x;
    jobs[3 * j + 1] = pr.y;
    jobs[3 * j + 2] = 0;
  }
}
__global__ void k_jobs_to_scores(const uint32_t* __restrict__ list, const uint32_t* __restrict__ bin_off,
                                 const uint32_t* __restrict__ bin_cnt, const uint32_t* __restrict__ jobs,
                                 uint32_t* __restrict__ score) {
  const uint32_t cnt = bin_cnt[kBinPlain], off = bin_off[kBinPlain];
  for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < cnt; j += gridDim.x * blockDim.x)
    score[list[off + j]] = jobs[3 * j + 2];
}
void plain_bin_jobs(const uint2* pairs, const uint32_t* list, const uint32_t* bin_off,
                    const uint32_t* bin_cnt, uint32_t* jobs, hipStream_t s) {
  hipLaunchKernelGGL(k_bin_to_jobs, dim3(64), dim3(256), 0, s, pairs, list, bin_off, bin_cnt, jobs);
  NGIA_HIP(hipGetLastError());
}
void plain_bin_scores(const uint32_t* list, const uint32_t* bin_off, const uint32_t* bin_cnt,
                      const uint32_t* jobs, uint32_t* score, hipStream_t s) {
  hipLaunchKernelGGL(k_jobs_to_scores, dim3(64), dim3(256), 0, s, list, bin_off, bin_cnt, jobs,
                     score);
  NGIA_HIP(hipGetLastError());
}

// Passing pairs -> raw edge list.  A block takes tiles of 4096 pairs (16 per
// thread), ranks its passing pairs with a block prefix sum and reserves their
// slots with one global atomic per tile: passing pairs are a few percent, and
// one atomic per wavefront on the shared counter serialised the kernel.  The
// list's order is free (the sort + unique follows).
__global__ __launch_bounds__(256) void k_pairs_to_edges(const uint2* __restrict__ pairs,
                                                        const uint64_t* __restrict__ npairs,
                                                        const uint32_t* __restrict__ score,
                                                        uint64_t* __restrict__ ekeys,
                                                        uint32_t* __restrict__ escores,
                                                        unsigned long long* __restrict__ ecount) {
  __shared__ uint32_t wsum[4];
  __shared__ unsigned long long bbase;
  const uint64_t P = *npairs;
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (uint64_t base = (uint64_t)blockIdx.x * 4096; base < P; base += (uint64_t)gridDim.x * 4096) {
    uint32_t sc[16], mine = 0;
    #pragma unroll
    for (int k = 0; k < 16; k++) {
      const uint64_t p = base + (uint64_t)k * 256 + tid;
      sc[k] = p < P ? score[p] : 0u;
      mine += sc[k] != 0u;
    }
    uint32_t x = mine;  // inclusive prefix over the wavefront
    #pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(x, o);
      if (lane >= (uint32_t)o) x += y;
    }
    if (lane == 63) wsum[wave] = x;
    __syncthreads();
    if (tid == 0) {
      uint32_t t = 0;
      for (int w = 0; w < 4; w++) {
        const uint32_t v = wsum[w];
        wsum[w] = t;
        t += v;
      }
      bbase = t ? atomicAdd(ecount, (unsigned long long)t) : 0ull;
    }
    __syncthreads();
    unsigned long long at = bbase + wsum[wave] + x - mine;
    #pragma unroll
    for (int k = 0; k < 16; k++) {
      if (sc[k] == 0u) continue;
      const uint2 pr = pairs[base + (uint64_t)k * 256 + tid];
      ekeys[at] = ((uint64_t)pr.x << 32) | pr.y;
      escores[at] = sc[k];
      at++;
    }
    __syncthreads();  // wsum and bbase are rewritten by the next tile
  }
}

void pairs_to_edges(const uint2* pairs, const uint64_t* npairs, const uint32_t* score,
                    uint64_t* ekeys, uint32_t* escores, unsigned long long* ecount, uint32_t grid,
                    hipStream_t s) {
  hipLaunchKernelGGL(k_pairs_to_edges, dim3(grid), dim3(256), 0, s, pairs, npairs, score, ekeys,
                     escores, ecount);
  NGIA_HIP(hipGetLastError());
}

// ------------------------------------------------------------- edge list
// The sorted edge list of a batched round, whose pairs are distinct: a counting
// sort by u, then each edge's place among its u's by the number of smaller v.
//  1. k_edge_count: a passing pair takes the next slot of its u (kept in
//     slot[p]) in degree[], zero beforehand (k_pair_count);
//  2. off = prefix sums of degree;
//  3. k_edge_scatter: its key and score to off[u] + slot;
//  4. k_edge_rank: from there to off[u] + its rank; its first block also writes
//     the rounds' counters to pinned memory.  Those were two copies, four with a
//     head; without them and the copy of the bin counts (k_bin_offsets) a step of
//     500 records takes 233 us instead of 249, of 10k 343 instead of 356, of 100k
//     1376 instead of 1393.
// The host reads no count in between.  A round with a u of more than kMaxDegree
// edges (max_degree says so; steps 3 and 4 return at once) is sorted by
// pairs_to_edges and finalize_edges instead, since a rank costs its u's degree.
// Rows of the bucketing give a u at most one edge per band; only a caller's own
// rows pass kMaxDegree.
// Bound: latency of a few dependent passes, and for the counting the atomics' round
// trip (16 in flight a thread: 200,000 16S reads, 6 million pairs, 80 us with
// four, 32 so).  Before: compaction, a host synchronisation, a radix or merge
// sort of the 64-bit keys and a unique pass with nothing to drop.  Kernels from
// the last score to the list: 10,000 proteins at -i 70 20 us in 6 (130 in 13
// with the gaps), 1 million at -i 50 180 us (430).
__global__ __launch_bounds__(256) void k_edge_count(const uint2* __restrict__ pairs,
                                                    const uint64_t* __restrict__ npairs,
                                                    const uint32_t* __restrict__ score,
                                                    uint32_t* __restrict__ degree,
                                                    uint32_t* __restrict__ slot,
                                                    unsigned long long* __restrict__ ecount,
                                                    unsigned long long* __restrict__ max_degree) {
  __shared__ uint32_t edges, over;
  if (threadIdx.x == 0) edges = over = 0;
  __syncthreads();
  const uint64_t P = *npairs;
  uint32_t mine = 0, most = 0;
  constexpr int kPer = 16;  // pairs a thread at a time; one at a time waits on memory for each
  for (uint64_t base = (uint64_t)blockIdx.x * 256 * kPer; base < P;
       base += (uint64_t)gridDim.x * 256 * kPer) {
    uint32_t u[kPer], on = 0;
    #pragma unroll
    for (int k = 0; k < kPer; k++) {
      const uint64_t p = base + (uint64_t)k * 256 + threadIdx.x;
      on |= (uint32_t)(p < P && score[p] != 0u) << k;
    }
    #pragma unroll
    for (int k = 0; k < kPer; k++)
      if (on >> k & 1) u[k] = pairs[base + (uint64_t)k * 256 + threadIdx.x].x;
    #pragma unroll
    for (int k = 0; k < kPer; k++)
      if (on >> k & 1) u[k] = atomicAdd(&degree[u[k]], 1u);
    #pragma unroll
    for (int k = 0; k < kPer; k++) {
      if (!(on >> k & 1)) continue;
      slot[base + (uint64_t)k * 256 + threadIdx.x] = u[k];
      most = u[k] + 1 > most ? u[k] + 1 : most;
    }
    mine += __popc(on);
  }
  for (int o = 32; o > 0; o >>= 1) mine += __shfl_xor(mine, o);
  if ((threadIdx.x & 63) == 0 && mine) atomicAdd(&edges, mine);
  if (most > kMaxDegree) atomicMax(&over, most);
  __syncthreads();
  if (threadIdx.x == 0 && edges) atomicAdd(ecount, (unsigned long long)edges);
  if (threadIdx.x == 0 && over) atomicMax(max_degree, (unsigned long long)over);
}

__global__ __launch_bounds__(256) void k_edge_scatter(const uint2* __restrict__ pairs,
                                                      const uint64_t* __restrict__ npairs,
                                                      const uint32_t* __restrict__ score,
                                                      const uint64_t* __restrict__ off,
                                                      const uint32_t* __restrict__ slot,
                                                      const unsigned long long* __restrict__ max_degree,
                                                      uint64_t* __restrict__ keys,
                                                      uint32_t* __restrict__ scores) {
  if (*max_degree > kMaxDegree) return;
  const uint64_t P = *npairs;
  for (uint64_t p = (uint64_t)blockIdx.x * 256 + threadIdx.x; p < P; p += (uint64_t)gridDim.x * 256) {
    const uint32_t sc = score[p];
    if (sc == 0) continue;
    const uint2 pr = pairs[p];
    const uint64_t at = off[pr.x] + slot[p];
    keys[at] = ((uint64_t)pr.x << 32) | pr.y;
    scores[at] = sc;
  }
}

__global__ __launch_bounds__(256) void k_edge_rank(RoundReport main, RoundReport head,
                                                   const uint64_t* __restrict__ off, uint32_t n,
                                                   const unsigned long long* __restrict__ max_degree,
                                                   const uint64_t* __restrict__ keys_in,
                                                   const uint32_t* __restrict__ scores_in,
                                                   uint64_t* __restrict__ keys,
                                                   uint32_t* __restrict__ scores) {
  if (blockIdx.x == 0) {
    for (const RoundReport* r : {&main, &head}) {
      if (!r->host) continue;
      for (uint32_t k = threadIdx.x; k < r->words; k += 256) r->host[k] = r->counters[k];
      if (threadIdx.x == 0) *r->host_pairs = *r->pairs;
    }
  }
  if (*max_degree > kMaxDegree) return;
  const uint64_t m = off[n];
  for (uint64_t e = (uint64_t)blockIdx.x * 256 + threadIdx.x; e < m; e += (uint64_t)gridDim.x * 256) {
    const uint64_t key = keys_in[e];
    const uint32_t sc = scores_in[e], u = (uint32_t)(key >> 32);
    const uint64_t first = off[u], end = off[u + 1];
    uint64_t at = first;
    for (uint64_t j = first; j < end; j++) at += keys_in[j] < key;
    keys[at] = key;
    scores[at] = sc;
  }
}

void edge_count(const uint2* pairs, const uint64_t* npairs, const uint32_t* score, uint32_t* degree,
                uint32_t* slot, unsigned long long* ecount, unsigned long long* max_degree,
                uint32_t grid, hipStream_t s) {
  hipLaunchKernelGGL(k_edge_count, dim3(grid), dim3(256), 0, s, pairs, npairs, score, degree, slot,
                     ecount, max_degree);
  NGIA_HIP(hipGetLastError());
}

void edge_scatter(const uint2* pairs, const uint64_t* npairs, const uint32_t* score,
                  const uint64_t* off, const uint32_t* slot, const unsigned long long* max_degree,
                  uint64_t* keys, uint32_t* scores, uint32_t grid, hipStream_t s) {
  hipLaunchKernelGGL(k_edge_scatter, dim3(grid), dim3(256), 0, s, pairs, npairs, score, off, slot,
                     max_degree, keys, scores);
  NGIA_HIP(hipGetLastError());
}

void edge_rank(const RoundReport& main, const RoundReport& head, const uint64_t* off, uint32_t n,
               const unsigned long long* max_degree, const uint64_t* keys_in,
               const uint32_t* scores_in, uint64_t* keys, uint32_t* scores, uint32_t grid,
               hipStream_t s) {
  hipLaunchKernelGGL(k_edge_rank, dim3(grid), dim3(256), 0, s, main, head, off, n, max_degree, keys_in,
                     scores_in, keys, scores);
  NGIA_HIP(hipGetLastError());
}

// Edges as the caller gets them, 12 bytes each, a word a thread.
__global__ __launch_bounds__(256) void k_edge_records(const uint64_t* __restrict__ keys,
                                                      const uint32_t* __restrict__ scores,
                                                      uint64_t m, uint32_t* __restrict__ out) {
  for (uint64_t t = (uint64_t)blockIdx.x * 256 + threadIdx.x; t < 3 * m; t += (uint64_t)gridDim.x * 256) {
    const uint64_t e = t / 3;
    const uint32_t k = (uint32_t)(t - 3 * e);
    out[t] = k == 0   ? (uint32_t)(keys[e] >> 32)
             : k == 1 ? (uint32_t)keys[e]
                      : __float_as_uint((float)scores[e] / 100.0f);  // buildGraph.hpp:346
  }
}

void edge_records(const uint64_t* keys, const uint32_t* scores, uint64_t m, uint32_t* out,
                  hipStream_t s) {
  if (m == 0) return;
  hipLaunchKernelGGL(k_edge_records, dim3((uint32_t)std::min<uint64_t>((3 * m + 255) / 256, 16384)),
                     dim3(256), 0, s, keys, scores, m, out);
  NGIA_HIP(hipGetLastError());
}

// ------------------------------------------------------------- finalize
// Sort the raw edges by (u,v) and drop duplicates (buildGraph.hpp:355-362):
// the score is a function of (u,v), so unique by key equals the reference's
// unique over (u,v,w) tuples.
size_t finalize_scratch_bytes(uint64_t m) {
  size_t a = 0, b = 0;
  (void)rocprim::radix_sort_pairs(nullptr, a, (uint64_t*)nullptr, (uint64_t*)nullptr,
                                  (uint32_t*)nullptr, (uint32_t*)nullptr, (size_t)m, 0, 64);
  (void)rocprim::unique_by_key(nullptr, b, (uint64_t*)nullptr, (uint32_t*)nullptr,
                               (uint64_t*)nullptr, (uint32_t*)nullptr,
                               (unsigned long long*)nullptr, (size_t)m);
  return (a > b ? a : b) + 256;
}

void finalize_edges(uint64_t* keys, uint32_t* scores, uint64_t m, uint32_t n, uint64_t* keys_tmp,
                    uint32_t* scores_tmp, void* temp, size_t temp_bytes,
                    unsigned long long* d_unique, hipStream_t s) {
  if (m == 0) {
    fill_u32((uint32_t*)d_unique, 0, 2, s);
    return;
  }
  // bits of the largest record index: the keys' bits from 32 + ib on are 0
  const uint32_t ib = n > 1 ? 32u - (uint32_t)__builtin_clz(n - 1) : 1u;
  size_t tb = temp_bytes;
  NGIA_HIP(rocprim::radix_sort_pairs(temp, tb, keys, keys_tmp, scores, scores_tmp, (size_t)m, 0,
                                     32 + ib, s));
  tb = temp_bytes;
  NGIA_HIP(rocprim::unique_by_key(temp, tb, keys_tmp, scores_tmp, keys, scores, d_unique, (size_t)m,
                                  rocprim::equal_to<uint64_t>(), s));
}

}  // namespace ngia
