// dev_sketch.hip -- minhash sketch (makedb.hpp:224-247) and band bucketing
// (makedb.hpp:289-364) on the device.
//
// Sketch mapping: one wavefront per sequence, lane k computes signature k.
// The 8-mer is the same for every lane, so it is built on the scalar unit
// from the sequence's byte codes (scalar loads, four codes per dword); the
// 64 hash functions run one per lane.  The first two steps of the hash fold:
// with h = kmer ^ seed_k,  (h ^ 61) ^ (h >> 16) =
//   (kmer ^ (kmer >> 16)) ^ (seed_k ^ 61 ^ (seed_k >> 16)),
// a wave-uniform term xor a per-lane constant, because a logical right shift
// distributes over xor.  Output is sequence-major: lane k of sequence i
// writes sig[64*i + k], one 256-byte coalesced store per wavefront.
#include <algorithm>
#include <cstring>
#include <type_traits>

#include <rocprim/rocprim.hpp>

#include "dev_common.hpp"
#include "dev_graph.hpp"

namespace ngia {

// The hash of an 8-mer (makedb.hpp:232-240): k1 = kmer ^ (kmer >> 16) and s1 the
// lane's seed term (below) carry its first two steps.
__device__ __forceinline__ uint32_t kmer_hash(uint32_t k1, uint32_t s1) {
  uint32_t h = k1 ^ s1;
  h = h + (h << 3);
  h = h ^ (h >> 4);
  h = h * 0x27d4eb2du;
  h = h ^ (h >> 15);
  h = (h ^ (h >> 8)) * 0x9e3779b1u;
  return h ^ (h >> 14);
}

// Hashes the windows ending at positions [j, end) of a record whose byte
// codes start at cw (four per dword), the k-mer of the positions before j in
// kmer; mn keeps the minimum.  Head to a 16-aligned position, then sixteen
// positions per four-dword scalar load: one wait on the scalar cache per
// sixteen windows.  The load reads whole 16-byte groups; a record's codes
// are padded to 32 bytes, so it stays within the record's own padding.
__device__ __forceinline__ void sketch_windows(const uint32_t* cw, uint32_t j, uint32_t end,
                                               uint32_t kmer, uint32_t s1, uint32_t& mn) {
  auto hash = [&](uint32_t k1) {
    const uint32_t h = kmer_hash(k1, s1);
    mn = h < mn ? h : mn;
  };
  for (; j < end && (j & 15); j++) {
    const uint32_t w = __builtin_amdgcn_readfirstlane(cw[j >> 2]);
    kmer = (kmer << 4) + ((w >> (8 * (j & 3))) & 0xFu);
    hash(kmer ^ (kmer >> 16));
  }
  for (; j + 16 <= end; j += 16) {
    const uint4 c4 = *(const uint4*)(cw + (j >> 2));
    const uint32_t ws[4] = {(uint32_t)__builtin_amdgcn_readfirstlane(c4.x),
                            (uint32_t)__builtin_amdgcn_readfirstlane(c4.y),
                            (uint32_t)__builtin_amdgcn_readfirstlane(c4.z),
                            (uint32_t)__builtin_amdgcn_readfirstlane(c4.w)};
    #pragma unroll
    for (int q = 0; q < 4; q++) {
      #pragma unroll
      for (int m = 0; m < 4; m++) {
        kmer = (kmer << 4) + ((ws[q] >> (8 * m)) & 0xFu);
        hash(kmer ^ (kmer >> 16));
      }
    }
  }
  for (; j + 4 <= end; j += 4) {
    const uint32_t w = __builtin_amdgcn_readfirstlane(cw[j >> 2]);
    #pragma unroll
    for (int m = 0; m < 4; m++) {
      kmer = (kmer << 4) + ((w >> (8 * m)) & 0xFu);
      hash(kmer ^ (kmer >> 16));
    }
  }
  for (; j < end; j++) {
    const uint32_t w = __builtin_amdgcn_readfirstlane(cw[j >> 2]);
    kmer = (kmer << 4) + ((w >> (8 * (j & 3))) & 0xFu);
    hash(kmer ^ (kmer >> 16));
  }
}

// The codes of record `seq` (the 64-bit offset moves to scalar registers as
// two halves: code areas pass 2^31 bytes at a few million sequences).
__device__ __forceinline__ const uint32_t* record_codes(const uint8_t* codes,
                                                        const uint64_t* code_off, uint32_t seq) {
  const uint64_t co = code_off[seq];
  const uint32_t co_lo = __builtin_amdgcn_readfirstlane((uint32_t)co);
  const uint32_t co_hi = __builtin_amdgcn_readfirstlane((uint32_t)(co >> 32));
  return (const uint32_t*)(codes + (((uint64_t)co_hi << 32) | co_lo));
}

// Hashing starts at position 7, or at the last position of a read shorter
// than 8 (makedb.hpp:234-235).
__device__ __forceinline__ uint32_t first_window(uint32_t L) { return L >= 8 ? 7u : (L ? L - 1 : 0u); }

// Lane k computes signature k: the per-lane half of the folded first two
// hash steps, seed_k ^ 61 ^ (seed_k >> 16).
__device__ __forceinline__ uint32_t lane_seed_term(uint32_t lane) {
  const uint32_t seed = lane * 0x9e3779b1u + 0x85ebca6bu;
  return seed ^ 61u ^ (seed >> 16);
}

// kList: the records list[0..n).
template <bool kList>
__global__ __launch_bounds__(256) void k_sketch(const uint8_t* __restrict__ codes,
                                                const uint64_t* __restrict__ code_off,
                                                const uint32_t* __restrict__ lengths,
                                                const uint32_t* __restrict__ list, uint32_t n,
                                                uint32_t* __restrict__ sig) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t item = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  if (item >= n) return;
  const uint32_t seq = kList ? __builtin_amdgcn_readfirstlane(list[item]) : item;
  const uint32_t L = __builtin_amdgcn_readfirstlane(lengths[seq]);
  const uint32_t* cw = record_codes(codes, code_off, seq);
  const uint32_t first = first_window(L);
  uint32_t kmer = 0;
  for (uint32_t j = 0; j < first; j++) {  // the prefix only feeds the k-mer
    const uint32_t w = __builtin_amdgcn_readfirstlane(cw[j >> 2]);
    kmer = (kmer << 4) + ((w >> (8 * (j & 3))) & 0xFu);
  }
  uint32_t mn = 0xFFFFFFFFu;
  sketch_windows(cw, first, L, kmer, lane_seed_term(lane), mn);
  sig[(uint64_t)seq * 64 + lane] = mn;
}

// Long records in pieces: one wavefront per (record, chunk of positions),
// chunks[c] = (record, first window position); a chunk ends at the next
// multiple of `len` or the record's end; the k-mer is rebuilt from the seven codes
// before the chunk (codes before position 0 count as 0, as in k_sketch).
// The minimum over a record's chunks is the same whatever their order:
// each wavefront folds its chunk's minima into sig with atomicMin, over
// signatures set to all ones first.
__global__ __launch_bounds__(256) void k_sketch_chunks(const uint8_t* __restrict__ codes,
                                                       const uint64_t* __restrict__ code_off,
                                                       const uint32_t* __restrict__ lengths,
                                                       const uint2* __restrict__ chunks,
                                                       uint32_t nchunks, uint32_t len,
                                                       uint32_t* __restrict__ sig) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t c = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  if (c >= nchunks) return;
  const uint2 ch = chunks[c];
  const uint32_t seq = __builtin_amdgcn_readfirstlane(ch.x);
  const uint32_t p0 = __builtin_amdgcn_readfirstlane(ch.y);
  const uint32_t L = __builtin_amdgcn_readfirstlane(lengths[seq]);
  const uint32_t* cw = record_codes(codes, code_off, seq);
  const uint32_t stop = p0 - p0 % len + len;
  const uint32_t end = stop < L ? stop : L;
  uint32_t kmer = 0;
  for (uint32_t j = p0 >= 7 ? p0 - 7 : 0u; j < p0; j++) {
    const uint32_t w = __builtin_amdgcn_readfirstlane(cw[j >> 2]);
    kmer = (kmer << 4) + ((w >> (8 * (j & 3))) & 0xFu);
  }
  uint32_t mn = 0xFFFFFFFFu;
  sketch_windows(cw, p0, end, kmer, lane_seed_term(lane), mn);
  atomicMin(&sig[(uint64_t)seq * 64 + lane], mn);
}

void launch_sketch_chunks(const uint8_t* codes, const uint64_t* code_off, const uint32_t* lengths,
                          const uint2* chunks, uint32_t nchunks, uint32_t len, uint32_t* sig,
                          hipStream_t stream) {
  if (nchunks == 0) return;
  hipLaunchKernelGGL(k_sketch_chunks, dim3((nchunks + 3) / 4), dim3(256), 0, stream, codes,
                     code_off, lengths, chunks, nchunks, len, sig);
  NGIA_HIP(hipGetLastError());
}

void launch_sketch(const uint8_t* codes, const uint64_t* code_off, const uint32_t* lengths,
                   uint32_t n, uint32_t* sig, hipStream_t stream, const uint32_t* list) {
  if (n == 0) return;
  if (list)
    hipLaunchKernelGGL(k_sketch<true>, dim3((n + 3) / 4), dim3(256), 0, stream, codes, code_off,
                       lengths, list, n, sig);
  else
    hipLaunchKernelGGL(k_sketch<false>, dim3((n + 3) / 4), dim3(256), 0, stream, codes, code_off,
                       lengths, list, n, sig);
  NGIA_HIP(hipGetLastError());
}

// ------------------------------------------------------- four-letter records
// A record over four letters (DNA) has at most 4^8 = 65,536 different 8-mers, so
// its signature in band b is the first 8-mer of the fixed list "all 8-mers by
// their band-b hash" that the record holds.  One wavefront marks the
// record's 8-mers in a bit set (8 KiB of LDS), then lane b walks down band b's
// list until it meets a marked one: with D different 8-mers about 65,536 / D
// probes on average (4.7 times that for the slowest of 64 lanes), in place of
// a hash per window.  Windows with any other letter (N, unknown ones) are
// hashed as before and join the minimum, one after another: a record with many of
// them, or a short one, is hashed throughout (walk_fits), here while such records
// are few, else by k_sketch.
// An 8-mer's place in the bit set comes from the records' bit planes: the two
// bits of a letter over 32 positions are two words, an 8-mer's bits eight
// consecutive ones of each.  A list entry holds the place as (byte address
// << 16 | bit), so that a probe is one shift, one LDS read, one shift and one
// v_alignbit that collects the hits of eight probes.
// The lists hold the smallest hashes only (about kWalkExpected of them: those
// below kWalkBound); a lane that reaches the end sends the record back to the
// plain loop, as do records whose D x length is below kWalkMin, where the walk
// is the longer way.
// Bound: VALU issue (1,290 instructions a record of 1,400 bases, 55% of the
// kernel's time) and waits on the list and the bit set at five wavefronts per
// SIMD.  Measured on 200,000 DNA records (280M bases): 4.77 ms with a hash per
// window, 0.71 ms here; 1.06 ms with the 8-mers rolled byte by byte and list
// entries unpacked per probe, 0.96 with one batch of eight probes in flight.
constexpr uint32_t kWalkExpected = 3072;
constexpr uint32_t kWalkBound = kWalkExpected << 16;
constexpr uint32_t kWalkCap = 4096;
constexpr uint32_t kWalkMin = 160000;

// The k-mer of codes of 8-mer idx: bits 0-7 hold the low bits of its letters in
// order, bits 8-15 the high bits; sym_code the code of letter y in bits 4y...
__device__ __forceinline__ uint32_t walk_kmer(uint32_t idx, uint32_t sym_code) {
  uint32_t kmer = 0;
  #pragma unroll
  for (int i = 0; i < 8; i++) {
    const uint32_t y = ((idx >> i) & 1u) | (((idx >> (8 + i)) & 1u) << 1);
    kmer = (kmer << 4) | ((sym_code >> (4 * y)) & 0xFu);
  }
  return kmer;
}

// Band blockIdx.x's list: entry t of band b at table[(t / 8) * 512 + b * 8 + t
// % 8].  *depth: the entries every band's list has (0: a list overflowed).
__global__ __launch_bounds__(1024) void k_walk_table(uint32_t sym_code, uint32_t* __restrict__ table,
                                                     uint32_t* __restrict__ depth) {
  using Sort = rocprim::block_radix_sort<uint32_t, 1024, kWalkCap / 1024, uint32_t>;
  __shared__ typename Sort::storage_type storage;
  __shared__ uint32_t hs[kWalkCap], ix[kWalkCap];
  __shared__ uint32_t cnt;
  const uint32_t b = blockIdx.x, t = threadIdx.x;
  if (t == 0) cnt = 0;
  __syncthreads();
  const uint32_t s1 = lane_seed_term(b);
  for (uint32_t i = t; i < 65536; i += 1024) {
    const uint32_t kmer = walk_kmer(i, sym_code);
    const uint32_t h = kmer_hash(kmer ^ (kmer >> 16), s1);
    if (h < kWalkBound) {
      const uint32_t at = atomicAdd(&cnt, 1u);
      if (at < kWalkCap) {
        hs[at] = h;
        ix[at] = i;
      }
    }
  }
  __syncthreads();
  const uint32_t n = cnt;
  if (n > kWalkCap) {
    if (t == 0) atomicMin(depth, 0u);
    return;
  }
  uint32_t key[kWalkCap / 1024], val[kWalkCap / 1024];
  #pragma unroll
  for (uint32_t j = 0; j < kWalkCap / 1024; j++) {
    const uint32_t q = t * (kWalkCap / 1024) + j;
    key[j] = q < n ? hs[q] : 0xFFFFFFFFu;
    val[j] = q < n ? ix[q] : 0u;
  }
  __syncthreads();
  Sort().sort(key, val, storage);
  #pragma unroll
  for (uint32_t j = 0; j < kWalkCap / 1024; j++) {
    const uint32_t q = t * (kWalkCap / 1024) + j;
    if (q < n) table[(q / 8) * 512 + b * 8 + (q & 7u)] = ((val[j] >> 5) << 18) | (val[j] & 31u);
  }
  if (t == 0) atomicMin(depth, n / 8 * 8);
}

size_t walk_table_bytes() { return (size_t)kWalkCap * 64 * 4 + 256; }

void launch_walk_table(uint32_t sym_code, void* table, hipStream_t stream) {
  uint32_t* depth = (uint32_t*)table + (size_t)kWalkCap * 64;
  fill_u32(depth, 0xFFFFFFFFu, 1, stream);
  hipLaunchKernelGGL(k_walk_table, dim3(64), dim3(1024), 0, stream, sym_code, (uint32_t*)table, depth);
  NGIA_HIP(hipGetLastError());
}

// The letters of a word of 32 positions: their low and high bits, and which
// positions hold one of the four.
struct LetterBits {
  uint32_t lo, hi, ok;
};
__device__ __forceinline__ LetterBits letter_bits(const uint32_t* pl, uint32_t sym_code) {
  const uint32_t p0 = pl[0], p1 = pl[1], p2 = pl[2], p3 = pl[3];
  uint32_t m[4];
  #pragma unroll
  for (int y = 0; y < 4; y++) {
    const uint32_t c = (sym_code >> (4 * y)) & 0xFu;
    const uint32_t x0 = (c & 1u) ? p0 : ~p0, x1 = (c & 2u) ? p1 : ~p1;
    const uint32_t x2 = (c & 4u) ? p2 : ~p2, x3 = (c & 8u) ? p3 : ~p3;
    m[y] = c ? x0 & x1 & x2 & x3 : 0u;  // code 0: the database has fewer letters
  }
  return {m[1] | m[3], m[2] | m[3], m[0] | m[1] | m[2] | m[3]};
}

// The positions of a block that end eight of the four letters in a row; p: the
// block before.
__device__ __forceinline__ uint32_t full_windows(uint32_t ok, uint32_t prev_ok) {
  uint64_t run = ((uint64_t)ok << 32) | prev_ok;
  run &= run << 1;
  run &= run << 2;
  run &= run << 4;
  return (uint32_t)(run >> 32);
}
// The positions of block blk that end a window of a record of L residues.
__device__ __forceinline__ uint32_t window_ends(uint32_t L, uint32_t blk) {
  const uint32_t left = L - 32 * blk;
  return (left < 32 ? (1u << left) - 1u : ~0u) & (blk ? ~0u : ~0x7Fu);
}

// others[i]: the windows of record i that hold another letter.  Four records a
// block, a wavefront each; bound by reading the records once, 4 bits a residue.
__global__ __launch_bounds__(256) void k_walk_others(const uint32_t* __restrict__ packed,
                                                     const uint64_t* __restrict__ word_off,
                                                     const uint32_t* __restrict__ lengths, uint32_t n,
                                                     uint32_t sym_code, uint32_t* __restrict__ others) {
  const uint32_t lane = threadIdx.x & 63u, seq = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (seq >= n) return;
  const uint32_t L = lengths[seq], nblk = (L + 31) / 32;
  const uint32_t* planes = packed + word_off[seq] + 1;
  uint32_t sum = 0;
  for (uint32_t blk = lane; blk < nblk; blk += 64) {
    const uint32_t ok = letter_bits(planes + 4ull * blk, sym_code).ok;
    const uint32_t prev = blk ? letter_bits(planes + 4ull * blk - 4, sym_code).ok : 0u;
    sum += __popc(~full_windows(ok, prev) & window_ends(L, blk));
  }
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
  if (lane == 0) others[seq] = sum;
}

void launch_walk_others(const uint32_t* packed, const uint64_t* word_off, const uint32_t* lengths,
                        uint32_t n, uint32_t sym_code, uint32_t* others, hipStream_t stream) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_walk_others, dim3((n + 3) / 4), dim3(256), 0, stream, packed, word_off, lengths,
                     n, sym_code, others);
  NGIA_HIP(hipGetLastError());
}

// sym_code: the code of letter y in bits 4y..; the records list[0..n), kHashRecord
// set in those to be hashed, or, without a list, 0..n-1.
__global__ __launch_bounds__(64) void k_sketch_walk(
    const uint32_t* __restrict__ packed, const uint64_t* __restrict__ word_off,
    const uint8_t* __restrict__ codes, const uint64_t* __restrict__ code_off,
    const uint32_t* __restrict__ lengths, const uint32_t* __restrict__ list, uint32_t n,
    uint32_t sym_code,
    const uint32_t* __restrict__ table, const uint32_t* __restrict__ depth,
    uint32_t* __restrict__ sig) {
  __shared__ __align__(16) uint32_t bits[2048];
  const uint32_t lane = threadIdx.x;
  const uint32_t s1 = lane_seed_term(lane);
  const uint32_t batches = *depth / 8;
  const uint4* const tab = (const uint4*)table + 2 * lane;  // batch q at tab[128 q], tab[128 q + 1]
  for (uint32_t item = blockIdx.x; item < n; item += gridDim.x) {
    const uint32_t entry = list ? __builtin_amdgcn_readfirstlane(list[item]) : item;
    const uint32_t seq = entry & ~kHashRecord;
    const uint32_t L = __builtin_amdgcn_readfirstlane(lengths[seq]);
    const uint32_t* cw = record_codes(codes, code_off, seq);
    uint32_t mn = 0xFFFFFFFFu;
    bool direct = (uint64_t)L * L < kWalkMin || entry != seq;
    if (!direct) {
      const uint32_t* planes = packed + word_off[seq] + 1;
      #pragma unroll
      for (int k = 0; k < 8; k++) ((uint4*)bits)[lane + 64 * k] = make_uint4(0u, 0u, 0u, 0u);
      __syncthreads();
      const uint32_t nblk = (L + 31) / 32;
      for (uint32_t b0 = 0; b0 < nblk; b0 += 64) {
        const uint32_t blk = b0 + lane;
        uint32_t other = 0;
        if (blk < nblk) {
          const LetterBits c = letter_bits(planes + 4ull * blk, sym_code);
          LetterBits pv = {0u, 0u, 0u};
          if (blk) pv = letter_bits(planes + 4ull * blk - 4, sym_code);
          const uint32_t ends = window_ends(L, blk), full = full_windows(c.ok, pv.ok) & ends;
          #pragma unroll
          for (int p = 0; p < 32; p++) {
            const uint32_t x = p < 7 ? __builtin_amdgcn_alignbit(c.lo, pv.lo, p + 25) : c.lo >> (p - 7);
            const uint32_t y = p < 7 ? __builtin_amdgcn_alignbit(c.hi, pv.hi, p + 25) : c.hi >> (p - 7);
            // bytes 0 of x and y
            const uint32_t idx = __builtin_amdgcn_perm(y, x, 0x0C0C0400u);
            atomicOr((uint32_t*)((char*)bits + ((idx >> 3) & 0x1FFCu)),
                     ((full >> p) & 1u) << (idx & 31u));
          }
          other = ~full & ends;
        }
        // windows with another letter, one at a time
        for (uint64_t who = __builtin_amdgcn_ballot_w64(other != 0); who; who &= who - 1) {
          const uint32_t src = (uint32_t)__builtin_ctzll(who);
          uint32_t m = __builtin_amdgcn_readlane(other, src);
          for (; m; m &= m - 1) {
            const uint32_t j = 32 * (b0 + src) + (uint32_t)__builtin_ctz(m);
            uint32_t kmer = 0;
            for (uint32_t q = j - 7; q <= j; q++) {
              const uint32_t w = __builtin_amdgcn_readfirstlane(cw[q >> 2]);
              kmer = (kmer << 4) + ((w >> (8 * (q & 3))) & 0xFu);
            }
            const uint32_t h = kmer_hash(kmer ^ (kmer >> 16), s1);
            mn = h < mn ? h : mn;
          }
        }
      }
      __syncthreads();
      uint32_t d = 0;
      #pragma unroll
      for (int k = 0; k < 8; k++) {
        const uint4 v = ((const uint4*)bits)[lane + 64 * k];
        d += __popc(v.x) + __popc(v.y) + __popc(v.z) + __popc(v.w);
      }
      for (int off = 32; off > 0; off >>= 1) d += __shfl_xor(d, off);
      direct = (uint64_t)d * L < kWalkMin || batches == 0;
    }
    if (!direct) {
      // Four batches are in flight: one at a time, a round waited for the
      // table (in L2) each eight probes.  A lane that has met its 8-mer leaves
      // the loop: the slowest lane probes 4.7 times as often as the average.
      uint32_t hit = 0, at = 0;
      uint4 e[4][2];
      #pragma unroll
      for (uint32_t u = 0; u < 4; u++) {
        const uint32_t nq = u < batches ? u : batches - 1;
        e[u][0] = tab[128 * nq];
        e[u][1] = tab[128 * nq + 1];
      }
      for (uint32_t q0 = 0; q0 < batches && !hit; q0 += 4) {
        #pragma unroll
        for (uint32_t u = 0; u < 4; u++) {
          const uint32_t w[8] = {e[u][0].x, e[u][0].y, e[u][0].z, e[u][0].w,
                                 e[u][1].x, e[u][1].y, e[u][1].z, e[u][1].w};
          const uint32_t nq = q0 + u + 4 < batches ? q0 + u + 4 : batches - 1;
          e[u][0] = tab[128 * nq];
          e[u][1] = tab[128 * nq + 1];
          uint32_t acc = 0;
          #pragma unroll
          for (int k = 0; k < 8; k++) {
            const uint32_t v = *(const uint32_t*)((const char*)bits + (w[k] >> 16));
            acc = __builtin_amdgcn_alignbit(v >> (w[k] & 31u), acc, 1);  // the probed bit enters on top
          }
          // past the last batch the last one is probed again: no hit there
          if (!hit) {
            hit = acc >> 24;
            at = q0 + u < batches ? q0 + u : batches - 1;
          }
        }
      }
      if (__builtin_amdgcn_ballot_w64(hit == 0) == 0) {
        const uint32_t e = table[at * 512 + lane * 8 + (uint32_t)__builtin_ctz(hit)];
        const uint32_t kmer = walk_kmer(((e >> 18) << 5) | (e & 31u), sym_code);
        const uint32_t h = kmer_hash(kmer ^ (kmer >> 16), s1);
        mn = h < mn ? h : mn;
      } else {
        direct = true;
      }
    }
    if (direct) {
      const uint32_t first = first_window(L);
      uint32_t kmer = 0;
      for (uint32_t j = 0; j < first; j++) {
        const uint32_t w = __builtin_amdgcn_readfirstlane(cw[j >> 2]);
        kmer = (kmer << 4) + ((w >> (8 * (j & 3))) & 0xFu);
      }
      sketch_windows(cw, first, L, kmer, s1, mn);
    }
    sig[(uint64_t)seq * 64 + lane] = mn;
    __syncthreads();  // the bit set is cleared by the next record
  }
}

void launch_sketch_walk(const uint32_t* packed, const uint64_t* word_off, const uint8_t* codes,
                        const uint64_t* code_off, const uint32_t* lengths, uint32_t n,
                        uint32_t sym_code, const void* table, uint32_t cus, uint32_t* sig,
                        hipStream_t stream, const uint32_t* list) {
  if (n == 0) return;
  const uint32_t* depth = (const uint32_t*)table + (size_t)kWalkCap * 64;
  // 20 wavefronts of 8 KiB per CU
  hipLaunchKernelGGL(k_sketch_walk, dim3(std::min(n, cus * 20u)), dim3(64), 0, stream, packed, word_off,
                     codes, code_off, lengths, list, n, sym_code, (const uint32_t*)table, depth, sig);
  NGIA_HIP(hipGetLastError());
}

// ------------------------------------------------------------- bucketing
// Per band the reference stable-sorts (sig, i) by sig (makedb.hpp:320-339)
// and points every element at its predecessor in the equal-signature run
// (makedb.hpp:340-347).  Here all 64 bands are sorted at once by a stable
// radix sort on the 32-bit signature alone, the value carrying (band, i)
// with the band in the top bits: the input is band-major with i ascending,
// so after the stable sort every equal-signature run lists its elements by
// band, then by i -- each band's run is a contiguous, i-ascending slice, and
// an element's predecessor is the previous element when that one has the
// same signature and the same band.  Rows start as the identity; only the
// non-head elements are scattered.  Values need n < 2^26; larger n uses the
// (band << 32 | sig) 38-bit key instead.
constexpr uint32_t kIdxBits = 26;
constexpr uint32_t kIdxMask = (1u << kIdxBits) - 1u;

__global__ __launch_bounds__(256) void k_bucket_keys(const uint32_t* __restrict__ sig, uint32_t n,
                                                     uint32_t* __restrict__ keys,
                                                     uint32_t* __restrict__ vals) {
  // 64 sequences x 64 bands tile through LDS: coalesced reads of the
  // sequence-major signatures, coalesced writes of band-major keys.
  __shared__ uint32_t tile[64][65];
  const uint32_t i0 = blockIdx.x * 64;
  const uint32_t t = threadIdx.x;
  for (uint32_t e = t; e < 64 * 64; e += 256) {
    const uint32_t si = e >> 6, b = e & 63;
    tile[si][b] = (i0 + si < n) ? sig[(uint64_t)(i0 + si) * 64 + b] : 0u;
  }
  __syncthreads();
  for (uint32_t e = t; e < 64 * 64; e += 256) {
    const uint32_t b = e >> 6, si = e & 63;
    const uint32_t i = i0 + si;
    if (i < n) {
      keys[(uint64_t)b * n + i] = tile[si][b];
      vals[(uint64_t)b * n + i] = (b << kIdxBits) | i;
    }
  }
}

__global__ __launch_bounds__(256) void k_rep_identity(uint32_t n, uint32_t* __restrict__ rep) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;  // blockIdx.y = band
  if (i < n) rep[(uint64_t)blockIdx.y * n + i] = i;
}

__global__ __launch_bounds__(256) void k_bucket_rep(const uint32_t* __restrict__ keys,
                                                    const uint32_t* __restrict__ vals,
                                                    uint64_t total, uint32_t n,
                                                    uint32_t* __restrict__ rep) {
  const uint64_t p = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (p == 0 || p >= total) return;
  const uint32_t v = vals[p], pv = vals[p - 1];
  if (keys[p] == keys[p - 1] && (v >> kIdxBits) == (pv >> kIdxBits))
    rep[(uint64_t)(v >> kIdxBits) * n + (v & kIdxMask)] = pv & kIdxMask;
}

// Wide form for n >= 2^26: keys (band << 32 | sig), values i.
__global__ __launch_bounds__(256) void k_bucket_keys_wide(const uint32_t* __restrict__ sig,
                                                          uint32_t n, uint64_t* __restrict__ keys,
                                                          uint32_t* __restrict__ vals) {
  const uint64_t e = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= (uint64_t)n * 64) return;
  const uint32_t b = (uint32_t)(e / n), i = (uint32_t)(e % n);
  keys[e] = ((uint64_t)b << 32) | sig[(uint64_t)i * 64 + b];
  vals[e] = i;
}

__global__ __launch_bounds__(256) void k_bucket_rep_wide(const uint64_t* __restrict__ keys,
                                                         const uint32_t* __restrict__ vals,
                                                         uint64_t total, uint32_t n,
                                                         uint32_t* __restrict__ rep) {
  const uint64_t p = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (p == 0 || p >= total) return;
  const uint64_t k = keys[p];
  if (keys[p - 1] == k) rep[(k >> 32) * n + vals[p]] = vals[p - 1];
}

// ------------------------------------------------ partitioned bucketing
// Only equality of signatures within a band matters, so the full sort above
// is replaced, for n <= kPartMaxN, by a partition and hash chains in LDS:
//  1. k_mix_columns: h = mix(sig), a bijection of the 32-bit signature that
//     spreads its bits (minhash values crowd near 0), band-major, and the rows
//     of bucket heads (their own index), which most elements are: k_part_chain
//     writes at random places, the others' rows only;
//  2. k_part_scatter: each band's (h, i) into 2^pb partitions by the top pb bits
//     of h, in no order.  A partition has room for kPartCap elements, twice or
//     more its average (pb is chosen for an average of 1,024 to 2,048);
//  3. k_part_chain: one block per partition hangs its elements into chains by
//     the low bits of h; each element walks its chain for the largest index
//     below its own with the same h, which is its predecessor in the
//     reference's stable (sig, i) order.
//  4. the host reads what is left (PartsLeft), as a rule nothing: partitions with
//     chains too long to walk go to k_part_few, or with more values to k_part_left,
//     which also takes those past their room (heavily repeated signatures), from the
//     column.
// Where that would take longer than the full sort, or a partition has more distinct
// values than it has room for, the host redoes the whole bucketing with the sort.
// Bound: memory for the first two, 4 + 8 and 4 + 8 bytes an element; the LDS's
// latency down the chains and the scattered 4-byte row writes for the third.
// Bands stay on one XCD (block b takes bands of XCD b mod 8), so that the short
// runs a partition and a row are written in meet in one L2.
// All 64 bands, against a radix sort by partition and a block sort for each, us:
//   records                       20,000  50,000  100,000  300,000     1M
//   random proteins                  392     422      464      666   1321
//                                     41      57       84      210    617
//   one signature set in 2%          393     424      598      963   3647
//                                    104     154      186      383   1161
//   in half of them                  554     603      777     1457   3600
//                                    121     236      402     1041   3000
//   in all                           261     310      468     1119   3178
//                                    168     255      412     1011   2938
//   1,000 copies of each             127     183      264      582   4587
//                                    133     189      294      691   3739
// (1M: k_mix_columns 121, k_part_scatter 224, k_part_chain 252; before steps 3 and 4
// bailed out and shared the work as they do, one set in all 9508, 1,000 copies 12058.)
constexpr uint32_t kPartMaxN = 2800000;
constexpr uint32_t kPartCap = 4096;
constexpr uint32_t kScatterTile = 8192, kScatterThreads = 1024;
constexpr uint32_t kPartMaxBits = 11;

// Partition bits for n records.
constexpr uint32_t part_bits(uint32_t n) {
  uint32_t pb = 0;
  while (pb < kPartMaxBits && (n >> pb) > kPartCap / 2) pb++;
  return pb;
}
static_assert(part_bits(kPartMaxN) <= kPartMaxBits && (kPartMaxN >> part_bits(kPartMaxN)) <= kPartCap / 2,
              "partitions too large at the largest n");

__device__ inline uint32_t sig_mix(uint32_t x) {
  x *= 0x9E3779B1u;  // odd multiplier: a bijection mod 2^32
  x ^= x >> 16;      // xor with a right shift of itself: a bijection
  x *= 0x85EBCA6Bu;
  x ^= x >> 13;
  return x;
}

__global__ __launch_bounds__(256) void k_mix_columns(const uint32_t* __restrict__ sig, uint32_t n,
                                                     uint32_t* __restrict__ col,
                                                     uint32_t* __restrict__ rep) {
  // 64 records x 64 bands through LDS, as in k_bucket_keys
  __shared__ uint32_t tile[64][65];
  const uint32_t i0 = blockIdx.x * 64;
  const uint32_t t = threadIdx.x;
  uint32_t v[16];  // all loads in flight before the first store
  #pragma unroll
  for (uint32_t k = 0; k < 16; k++) {
    const uint32_t e = t + 256 * k;
    v[k] = sig[i0 + (e >> 6) < n ? (uint64_t)(i0 + (e >> 6)) * 64 + (e & 63) : 0u];
  }
  #pragma unroll
  for (uint32_t k = 0; k < 16; k++) tile[(t + 256 * k) >> 6][t & 63] = v[k];
  __syncthreads();
  for (uint32_t e = t; e < 64 * 64; e += 256) {
    const uint32_t b = e >> 6, si = e & 63;
    if (i0 + si < n) {
      col[(uint64_t)b * n + i0 + si] = sig_mix(tile[si][b]);
      rep[(uint64_t)b * n + i0 + si] = i0 + si;
    }
  }
}

// The band and the place within the band of a block, bands spread over the
// XCDs: blocks of bands 8x .. 8x + 7 run on XCD x, band by band.
__device__ inline void band_block(uint32_t per_band, uint32_t* band, uint32_t* at) {
  const uint32_t q = blockIdx.x / 8;
  *band = (blockIdx.x % 8) * 8 + q / per_band;
  *at = q % per_band;
}

// One tile of a band's column: counted by partition, given room by one atomic
// per partition, ordered by partition in LDS, written as runs.
__global__ __launch_bounds__(kScatterThreads) void k_part_scatter(const uint32_t* __restrict__ col, uint32_t n,
                                                      uint32_t pb, uint32_t tiles,
                                                      uint32_t* __restrict__ cursor,
                                                      uint2* __restrict__ entries) {
  __shared__ __align__(16) uint2 stage[kScatterTile];
  __shared__ uint32_t cnt[1u << kPartMaxBits], base[1u << kPartMaxBits];
  __shared__ uint32_t wsum[kScatterThreads / 64];
  constexpr uint32_t kPer = (1u << kPartMaxBits) / kScatterThreads;  // partitions a thread
  constexpr uint32_t kItems = kScatterTile / kScatterThreads;
  const uint32_t t = threadIdx.x, parts = 1u << pb;
  uint32_t band, tile;
  band_block(tiles, &band, &tile);
  const uint32_t i0 = tile * kScatterTile;
  const uint32_t m = n - i0 < kScatterTile ? n - i0 : kScatterTile;
  for (uint32_t k = t; k < parts; k += kScatterThreads) cnt[k] = 0;
  __syncthreads();
  uint32_t h[kItems], r[kItems];
  #pragma unroll
  for (uint32_t j = 0; j < kItems; j++) {
    const uint32_t q = j * kScatterThreads + t;
    h[j] = q < m ? col[(uint64_t)band * n + i0 + q] : 0u;
  }
  // pb = 0: a shift by 32 would be none
  auto part_of = [&](uint32_t x) { return (uint32_t)(((uint64_t)x << pb) >> 32); };
  #pragma unroll
  for (uint32_t j = 0; j < kItems; j++)
    if (j * kScatterThreads + t < m) r[j] = atomicAdd(&cnt[part_of(h[j])], 1u);
  __syncthreads();
  // exclusive prefix over the partitions
  const uint32_t k0 = kPer * t;
  uint32_t c[kPer], sum = 0;
  #pragma unroll
  for (uint32_t k = 0; k < kPer; k++) {
    c[k] = k0 + k < parts ? cnt[k0 + k] : 0u;
    sum += c[k];
  }
  uint32_t x = sum;
  #pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, o);
    if ((t & 63) >= (uint32_t)o) x += y;
  }
  if ((t & 63) == 63) wsum[t >> 6] = x;
  __syncthreads();
  uint32_t run = x - sum;
  for (uint32_t w = 0; w < t >> 6; w++) run += wsum[w];
  #pragma unroll
  for (uint32_t k = 0; k < kPer; k++) {
    if (k0 + k >= parts) break;
    const uint32_t g = c[k] ? atomicAdd(&cursor[(band << pb) + k0 + k], c[k]) : 0u;
    cnt[k0 + k] = run;
    base[k0 + k] = g - run;  // place in the partition of the tile's element s: base + s
    run += c[k];
  }
  __syncthreads();
  #pragma unroll
  for (uint32_t j = 0; j < kItems; j++)
    if (j * kScatterThreads + t < m) stage[cnt[part_of(h[j])] + r[j]] = make_uint2(h[j], i0 + j * kScatterThreads + t);
  __syncthreads();
  for (uint32_t q = t; q < m; q += kScatterThreads) {
    const uint2 e = stage[q];
    const uint32_t k = part_of(e.x), at = base[k] + q;
    if (at < kPartCap) entries[(uint64_t)((band << pb) + k) * kPartCap + at] = e;
  }
}

// The rows of `cnt` elements (h, i) in LDS, in any order: chained through next[]
// by the low bits of h (a chain ends at element kPartCap, which matches
// nothing and follows itself), a row written for every
// element with a predecessor.  A walk takes kChainMax steps at most; past that
// *many is set and the rows are left to k_part_left, at once where the chains are
// longer than kChainMean on average.  *chains: 0.
constexpr uint32_t kChainMax = 96, kChainMean = 64;
// A thread walks the chains of all its elements in step: one after another, each
// would wait for the longest chain of its wavefront.
constexpr uint32_t kHeads = 2048;
template <int BS, int kItems>
__device__ inline void chain_rows(uint2* el, uint16_t* next, uint32_t* head, uint32_t cnt,
                                  uint32_t* __restrict__ rep, uint32_t* many, uint32_t* chains) {
  const uint32_t t = threadIdx.x;
  #pragma unroll
  for (uint32_t k = 0; k < kHeads / BS; k++) head[t + k * BS] = kPartCap;
  if (t == 0) {
    el[kPartCap] = make_uint2(~0u, ~0u);
    next[kPartCap] = (uint16_t)kPartCap;
  }
  __syncthreads();
  uint32_t h[kItems], i[kItems], f[kItems], best[kItems];  // best: the predecessor's index + 1
  #pragma unroll
  for (int j = 0; j < kItems; j++) {
    const uint32_t e = t + j * BS;
    const uint2 x = el[e < cnt ? e : kPartCap];
    h[j] = x.x;
    i[j] = x.y;
    best[j] = 0;
  }
  uint32_t firsts = 0;  // the wavefront's elements that start a chain
  #pragma unroll
  for (int j = 0; j < kItems; j++) {
    const uint32_t e = t + j * BS;
    uint32_t f = 0;
    if (e < cnt) {
      f = atomicExch(&head[h[j] % kHeads], e);
      next[e] = (uint16_t)f;
    }
    firsts += (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(f == kPartCap));
  }
  if ((t & 63) == 0) atomicAdd(chains, firsts);
  __syncthreads();
  if (cnt > kChainMean * *chains) {
    if (t == 0) *many = 1u;
    __syncthreads();
    return;
  }
  #pragma unroll
  for (int j = 0; j < kItems; j++) f[j] = t + j * BS < cnt ? head[h[j] % kHeads] : kPartCap;
  bool more = true;
  for (uint32_t steps = 0; more && steps < kChainMax; steps++) {
    uint2 x[kItems];
    #pragma unroll
    for (int j = 0; j < kItems; j++) {
      x[j] = el[f[j]];
      f[j] = next[f[j]];
    }
    more = false;
    #pragma unroll
    for (int j = 0; j < kItems; j++) {
      if (x[j].x == h[j] && x[j].y < i[j] && x[j].y + 1 > best[j]) best[j] = x[j].y + 1;
      more = more || f[j] != kPartCap;
    }
  }
  if (more) *many = 1u;
  #pragma unroll
  for (int j = 0; j < kItems; j++)
    if (best[j] && f[j] == kPartCap) rep[i[j]] = best[j] - 1;
  __syncthreads();
}

constexpr uint32_t kRanges = 2048;
// Exclusive prefix sums of count[0..kRanges) in place, count[kRanges] the total.
template <int BS>
__device__ inline void range_starts(uint32_t* count, uint32_t* wsum) {
  constexpr uint32_t kPer = kRanges / BS;
  const uint32_t t = threadIdx.x;
  uint32_t c[kPer], sum = 0;
  #pragma unroll
  for (uint32_t k = 0; k < kPer; k++) {
    c[k] = count[t * kPer + k];
    sum += c[k];
  }
  uint32_t run = sum;
  #pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(run, o);
    if ((t & 63) >= (uint32_t)o) run += y;
  }
  if ((t & 63) == 63) wsum[t >> 6] = run;
  __syncthreads();
  run -= sum;
  for (uint32_t w = 0; w < t >> 6; w++) run += wsum[w];
  #pragma unroll
  for (uint32_t k = 0; k < kPer; k++) {
    count[t * kPer + k] = run;
    run += c[k];
  }
  if (t == BS - 1) count[kRanges] = run;
  __syncthreads();
}

// The elements of a partition in LDS brought into index order: counted and placed
// by 2,048 ranges of indices, then each by its rank within its range, which holds
// few elements, and at most n / 2048.  start: 2,049 words.
template <int BS, int kItems>
__device__ inline void index_order(uint2* el, uint32_t cnt, uint32_t n, uint32_t* start, uint32_t* wsum) {
  const uint32_t t = threadIdx.x;
  const uint32_t bits = n > 1 ? 32u - (uint32_t)__builtin_clz(n - 1) : 1u;
  const uint32_t shift = bits > 11 ? bits - 11 : 0u;
  for (uint32_t k = t; k < kRanges; k += BS) start[k] = 0;
  __syncthreads();
  uint2 x[kItems];
  uint32_t r[kItems];
  #pragma unroll
  for (int j = 0; j < kItems; j++) {
    const uint32_t e = t + j * BS;
    if (e < cnt) {
      x[j] = el[e];
      r[j] = atomicAdd(&start[x[j].y >> shift], 1u);
    }
  }
  __syncthreads();
  range_starts<BS>(start, wsum);
  #pragma unroll
  for (int j = 0; j < kItems; j++)
    if (t + j * BS < cnt) el[start[x[j].y >> shift] + r[j]] = x[j];
  __syncthreads();
  #pragma unroll
  for (int j = 0; j < kItems; j++) {
    if (t + j * BS >= cnt) continue;
    const uint32_t first = start[x[j].y >> shift], end = start[(x[j].y >> shift) + 1];
    r[j] = first;
    for (uint32_t e = first; e < end; e++) r[j] += el[e].y < x[j].y;
  }
  __syncthreads();
  #pragma unroll
  for (int j = 0; j < kItems; j++)
    if (t + j * BS < cnt) el[r[j]] = x[j];
  __syncthreads();
}

// The rows of a partition of at most kFewMax values: its elements by value and,
// within one, by ranges between its first and its last index, in kRanges ranges in
// all.  An element's predecessor is the largest index below its own in its range or,
// without one, the largest of the nearest range below that holds any.  False (and
// nothing written) with more values, or more than kFewCrowd elements in a range.
constexpr uint32_t kFewMax = 64, kFewSlots = 256, kFewCrowd = 128;
struct FewValues {
  uint32_t table[kFewSlots];  // 0, or an element of the slot's value, plus one
  uint32_t id[kFewSlots];     // the slots in use, counted
  uint32_t low[kFewMax], high[kFewMax], scale[kFewMax];
  uint32_t values, crowded;
};
template <int BS, int kItems>
__device__ inline bool few_rows(uint2* el, uint32_t cnt, uint32_t* __restrict__ rep, uint32_t* start,
                                uint32_t* wsum, FewValues& few) {
  const uint32_t t = threadIdx.x;
  for (uint32_t k = t; k < kRanges; k += BS) start[k] = 0;
  for (uint32_t k = t; k < kFewSlots; k += BS) few.table[k] = 0;
  if (t < kFewMax) {
    few.low[t] = ~0u;
    few.high[t] = 0;
  }
  if (t == 0) few.values = few.crowded = 0;
  __syncthreads();
  uint2 x[kItems];
  uint32_t v[kItems], r[kItems];  // value, place in its range
  #pragma unroll
  for (int j = 0; j < kItems; j++) {
    const uint32_t e = t + j * BS;
    x[j] = el[e < cnt ? e : 0];
    uint32_t s = x[j].x % kFewSlots;
    // ends at a slot of the value's own, or once there are too many values
    while (e < cnt && __hip_atomic_load(&few.values, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) <= kFewMax) {
      uint32_t was = __hip_atomic_load(&few.table[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (was == 0) was = atomicCAS(&few.table[s], 0u, e + 1);
      if (was == 0) atomicAdd(&few.values, 1u);
      if (was == 0 || el[was - 1].x == x[j].x) break;
      s = (s + 1) % kFewSlots;
    }
    v[j] = s;
  }
  __syncthreads();
  const uint32_t values = few.values;
  if (values > kFewMax) return false;
  if (t < kFewSlots) {
    const bool used = few.table[t] != 0;
    const uint64_t m = __builtin_amdgcn_ballot_w64(used);
    if ((t & 63) == 0) wsum[t >> 6] = (uint32_t)__popcll(m);
    few.id[t] = (uint32_t)__popcll(m & ((1ull << (t & 63)) - 1ull));
  }
  __syncthreads();
  #pragma unroll
  for (int j = 0; j < kItems; j++) {
    if (t + j * BS >= cnt) continue;
    uint32_t id = few.id[v[j]];
    for (uint32_t w = 0; w < v[j] >> 6; w++) id += wsum[w];
    v[j] = id;
    // most do not change them: all at one address, atomics take turns
    if (x[j].y < __hip_atomic_load(&few.low[id], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP))
      atomicMin(&few.low[id], x[j].y);
    if (x[j].y > __hip_atomic_load(&few.high[id], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP))
      atomicMax(&few.high[id], x[j].y);
  }
  __syncthreads();
  const uint32_t ranges = kRanges / values;  // of a value
  if (t < values) {
    const uint32_t span = few.high[t] - few.low[t] + 1;
    const uint32_t use = ranges < span ? ranges : span - 1;  // the product stays below it
    few.scale[t] = (uint32_t)(((uint64_t)use << 32) / span);
  }
  __syncthreads();
  auto range_of = [&](uint32_t id, uint32_t i) {
    return id * ranges + __umulhi(i - few.low[id], few.scale[id]);
  };
  #pragma unroll
  for (int j = 0; j < kItems; j++) {
    if (t + j * BS >= cnt) continue;
    r[j] = atomicAdd(&start[range_of(v[j], x[j].y)], 1u);
    if (r[j] >= kFewCrowd) few.crowded = 1;
  }
  __syncthreads();
  if (few.crowded) return false;
  range_starts<BS>(start, wsum);
  #pragma unroll
  for (int j = 0; j < kItems; j++)
    if (t + j * BS < cnt) el[start[range_of(v[j], x[j].y)] + r[j]] = x[j];
  __syncthreads();
  #pragma unroll
  for (int j = 0; j < kItems; j++) {
    if (t + j * BS >= cnt) continue;
    const uint32_t k = range_of(v[j], x[j].y), first = start[k];
    uint32_t best = 0;  // the predecessor's index + 1
    for (uint32_t e = first; e < start[k + 1]; e++)
      if (el[e].y < x[j].y && el[e].y + 1 > best) best = el[e].y + 1;
    if (!best && first > start[v[j] * ranges])
      for (uint32_t e = start[range_of(v[j], el[first - 1].y)]; e < first; e++)
        best = el[e].y + 1 > best ? el[e].y + 1 : best;
    if (best) rep[x[j].y] = best - 1;
  }
  return true;
}

// Elements in index order sorted in LDS, stably, by the bits of h below the
// partition's pb; an element's predecessor is the one before it if that has the same
// h.  kKeep: leaves the last element of each value in el[] and returns how many
// these are.  The sort's storage overlays the elements.
template <int BS, int kItems>
constexpr size_t kSortBytes =
    std::max(sizeof(typename rocprim::block_radix_sort<uint32_t, BS, kItems, uint32_t>::storage_type),
             (size_t)8 * BS * kItems);
template <int BS, int kItems, bool kKeep>
__device__ inline uint32_t sort_rows(uint2* el, uint32_t cnt, uint32_t pb, uint32_t* __restrict__ rep,
                                     uint32_t* wsum) {
  using Sort = rocprim::block_radix_sort<uint32_t, BS, kItems, uint32_t>;
  static_assert(kSortBytes<BS, kItems> <= kSortBytes<BS, (int)kPartCap / BS>, "more than the room");
  auto& storage = *reinterpret_cast<typename Sort::storage_type*>(el);
  const uint32_t t = threadIdx.x;
  uint32_t key[kItems], val[kItems];
  #pragma unroll
  for (int j = 0; j < kItems; j++) {
    const uint32_t q = t * kItems + j;
    const uint2 x = q < cnt ? el[q] : make_uint2(~0u, ~0u);  // the padding stays last
    key[j] = x.x;
    val[j] = x.y;
  }
  __syncthreads();
  Sort().sort(key, val, storage, 0, 32 - pb);
  __syncthreads();
  el[t] = make_uint2(key[kItems - 1], val[kItems - 1]);
  el[BS + t] = make_uint2(key[0], 0);
  __syncthreads();
  uint2 prev = t ? el[t - 1] : make_uint2(~key[0], 0);
  const uint32_t after = t + 1 < BS ? el[BS + t + 1].x : 0u;  // no element past the last thread's
  uint32_t keep = 0;  // bit j: the last element of its value
  #pragma unroll
  for (int j = 0; j < kItems; j++) {
    const uint32_t q = t * kItems + j;
    if (q < cnt && prev.x == key[j]) rep[val[j]] = prev.y;
    prev = make_uint2(key[j], val[j]);
    const uint32_t h = j + 1 < kItems ? key[j + 1 < kItems ? j + 1 : j] : after;
    if (q < cnt && (q + 1 == cnt || h != key[j])) keep |= 1u << j;
  }
  if (!kKeep) return 0;
  uint32_t x = __popc(keep);
  #pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, o);
    if ((t & 63) >= (uint32_t)o) x += y;
  }
  if ((t & 63) == 63) wsum[t >> 6] = x;
  __syncthreads();
  uint32_t at = x - __popc(keep), total = 0;
  for (uint32_t w = 0; w < BS / 64; w++) {
    if (w < t >> 6) at += wsum[w];
    total += wsum[w];
  }
  #pragma unroll
  for (int j = 0; j < kItems; j++)
    if (keep >> j & 1) el[at++] = make_uint2(key[j], val[j]);
  __syncthreads();
  return total;
}

// The rows of a partition of any size, from the band's whole column: its
// elements in index order, as many at a time as the room holds, behind the
// last element of each value so far.  False when these leave no room.
// Bound: a round trip to the column for every 4,096 of its elements, asked for a
// round ahead (one barrier each; one for every 512 took 0.9 ns an element), and a
// sort for every 4,096 that are the partition's.
template <int BS>
__device__ inline bool long_rows(const uint32_t* __restrict__ col, uint32_t n, uint32_t pb,
                                 uint32_t part, uint2* el, uint32_t* __restrict__ rep,
                                 uint32_t (*wsum)[BS / 64], uint32_t* keep_sum) {
  constexpr uint32_t kLoads = 8;
  constexpr int kItems = (int)kPartCap / BS;
  const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
  const uint32_t mine = w * 64 * kLoads + lane;  // a wavefront's elements lie together
  uint32_t cnt = 0, h[kLoads], next[kLoads];
  #pragma unroll
  for (uint32_t k = 0; k < kLoads; k++) next[k] = mine + 64 * k < n ? col[mine + 64 * k] : 0u;
  __syncthreads();
  for (uint32_t q0 = 0, round = 0; q0 < n; q0 += kLoads * BS, round ^= 1) {
    uint64_t m[kLoads];
    uint32_t own = 0;  // of the wavefront
    #pragma unroll
    for (uint32_t k = 0; k < kLoads; k++) {
      h[k] = next[k];
      const uint32_t i = q0 + mine + 64 * k, j = i + kLoads * BS;
      next[k] = j < n ? col[j] : 0u;
      m[k] = __builtin_amdgcn_ballot_w64(i < n && (uint32_t)(((uint64_t)h[k] << pb) >> 32) == part);
      own += (uint32_t)__popcll(m[k]);
    }
    if (lane == 0) wsum[round][w] = own;
    __syncthreads();
    uint32_t total = 0, before = 0;
    for (uint32_t v = 0; v < BS / 64; v++) {
      if (v < w) before += wsum[round][v];
      total += wsum[round][v];
    }
    auto put = [&](uint32_t at) {
      #pragma unroll
      for (uint32_t k = 0; k < kLoads; k++) {
        if ((m[k] >> lane) & 1ull)
          el[at + (uint32_t)__popcll(m[k] & ((1ull << lane) - 1ull))] = make_uint2(h[k], q0 + mine + 64 * k);
        at += (uint32_t)__popcll(m[k]);
      }
    };
    if (cnt + total <= kPartCap) {  // the same in every thread
      put(cnt + before);
      cnt += total;
      continue;
    }
    // else a wavefront's at a time, sorting in between
    for (uint32_t v = 0; v < BS / 64; v++) {
      const uint32_t some = wsum[round][v];
      if (cnt + some > kPartCap) {
        __syncthreads();
        cnt = sort_rows<BS, kItems, true>(el, cnt, pb, rep, keep_sum);
        if (cnt + 64 * kLoads > kPartCap) return false;
      }
      if (v == w) put(cnt);
      cnt += some;
    }
  }
  __syncthreads();
  sort_rows<BS, kItems, false>(el, cnt, pb, rep, keep_sum);
  return true;
}

// What k_part_chain leaves, for each XCD's eight bands a run of `list`: from its
// front the partitions with a long chain, from its end those with more elements
// than room, whose elements are `most` at most and `elements` in all.  overflow:
// those of them that had too many values.
struct PartsLeft {
  uint32_t overflow, most, elements;
  uint32_t sorts[8], longs[8];
};
static_assert(sizeof(PartsLeft) <= kBucketPinned, "no room in pinned memory");

__global__ __launch_bounds__(512) void k_part_chain(const uint2* __restrict__ entries,
                                                    const uint32_t* __restrict__ cursor, uint32_t n,
                                                    uint32_t pb, uint32_t* __restrict__ rep,
                                                    PartsLeft* __restrict__ left,
                                                    uint32_t* __restrict__ list) {
  __shared__ __align__(16) uint2 el[kPartCap + 2];
  __shared__ uint32_t head[kHeads], many, chains;
  __shared__ uint16_t next[kPartCap + 2];
  uint32_t band, at;
  band_block(1u << pb, &band, &at);
  const uint32_t part = (band << pb) + at, cnt = cursor[part];
  const uint32_t x = band / 8, run = 8u << pb;
  if (cnt > kPartCap) {
    if (threadIdx.x == 0) {
      list[(x + 1) * run - 1 - atomicAdd(&left->longs[x], 1u)] = part;
      atomicMax(&left->most, cnt);
      atomicAdd(&left->elements, cnt);
    }
    return;
  }
  if (threadIdx.x == 0) many = chains = 0;
  const uint2* const v = entries + (uint64_t)part * kPartCap;
  for (uint32_t e = threadIdx.x; e < cnt; e += 512) el[e] = v[e];
  __syncthreads();
  uint32_t* const row = rep + (uint64_t)band * n;
  // most partitions hold half the room: four elements a thread, not eight
  if (cnt <= kPartCap / 2)
    chain_rows<512, (int)kPartCap / 1024>(el, next, head, cnt, row, &many, &chains);
  else
    chain_rows<512, (int)kPartCap / 512>(el, next, head, cnt, row, &many, &chains);
  if (threadIdx.x == 0 && many) list[x * run + atomicAdd(&left->sorts[x], 1u)] = part;
}

// The partitions with a long chain that few_rows takes: their entries in the list
// become kDone.  Blocks keep to their XCD's bands, as before.  Bound: latency, three
// blocks a CU; the next partition's place and size are asked for a round ahead.
constexpr uint32_t kDone = ~0u;
constexpr uint32_t kFewBlocks = 768;
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(6, 6))) void k_part_few(
    const PartsLeft* __restrict__ left, uint32_t* __restrict__ list, const uint2* __restrict__ entries,
    const uint32_t* __restrict__ cursor, uint32_t n, uint32_t pb, uint32_t* __restrict__ rep) {
  __shared__ __align__(16) uint2 el[kPartCap];
  __shared__ uint32_t start[kRanges + 1], sums[8];
  __shared__ FewValues few;
  const uint32_t x = blockIdx.x % 8, run = 8u << pb, sorts = left->sorts[x], step = gridDim.x / 8;
  uint32_t p = blockIdx.x / 8;
  if (p >= sorts) return;
  uint32_t part = list[x * run + p], cnt = cursor[part];
  for (; p < sorts; p += step) {
    const uint32_t after = p + step < sorts ? p + step : p;
    const uint32_t next = list[x * run + after], next_cnt = cursor[next];
    uint32_t* const row = rep + (uint64_t)(part >> pb) * n;
    const uint2* const v = entries + (uint64_t)part * kPartCap;
    __syncthreads();
    for (uint32_t e = threadIdx.x; e < cnt; e += 512) el[e] = v[e];
    __syncthreads();
    // two or four elements a thread for most partitions
    const bool ok = cnt <= 1024   ? few_rows<512, 2>(el, cnt, row, start, sums, few)
                    : cnt <= 2048 ? few_rows<512, 4>(el, cnt, row, start, sums, few)
                                  : few_rows<512, 8>(el, cnt, row, start, sums, few);
    if (ok && threadIdx.x == 0) list[x * run + p] = kDone;
    part = next;
    cnt = next_cnt;
  }
}

// The others: those past their room, the longest work, from the column, then the
// rest sorted.  A kernel of its own for the sort's registers, which would cost
// k_part_chain a third of its wavefronts (1M records: 940 us against 840).
__global__ __launch_bounds__(512) void k_part_left(PartsLeft* __restrict__ left,
                                                   const uint32_t* __restrict__ list,
                                                   const uint2* __restrict__ entries,
                                                   const uint32_t* __restrict__ cursor,
                                                   const uint32_t* __restrict__ col, uint32_t n,
                                                   uint32_t pb, uint32_t* __restrict__ rep) {
  constexpr int kItems = (int)kPartCap / 512;
  __shared__ __align__(16) unsigned char mem[kSortBytes<512, kItems>];
  __shared__ uint32_t start[kRanges + 1], wsum[2][8], sums[8];
  uint2* const el = (uint2*)mem;
  const uint32_t x = blockIdx.x % 8, run = 8u << pb;
  const uint32_t longs = left->longs[x], sorts = left->sorts[x];
  for (uint32_t p = blockIdx.x / 8; p < longs + sorts; p += gridDim.x / 8) {
    const uint32_t part = list[p < longs ? (x + 1) * run - 1 - p : x * run + p - longs];
    if (part == kDone) continue;
    const uint32_t cnt = cursor[part];
    const uint64_t row = (uint64_t)(part >> pb) * n;
    __syncthreads();
    if (p < longs) {
      if (!long_rows<512>(col + row, n, pb, part & ((1u << pb) - 1u), el, rep + row, wsum, sums) &&
          threadIdx.x == 0)
        atomicAdd(&left->overflow, 1u);
      continue;
    }
    const uint2* const v = entries + (uint64_t)part * kPartCap;
    for (uint32_t e = threadIdx.x; e < cnt; e += 512) el[e] = v[e];
    __syncthreads();
    index_order<512, kItems>(el, cnt, n, start, sums);
    sort_rows<512, kItems, false>(el, cnt, pb, rep + row, sums);
  }
}

// Bucketing of at most kBucketSmallMax records (the head of a step, and any
// database that small), with no host synchronisation, so that it runs beside
// other kernels.
//
// Up to kMapMin records one block per band sorts the band's n (mix(sig), i)
// pairs in LDS, stably, and points each element equal to its predecessor at
// that predecessor.  The sort's storage holds the threads' last items after
// the sort (8 bytes per thread, well inside it).
constexpr uint32_t kMapMin = 8192;
template <int BS, int ITEMS>
__global__ __launch_bounds__(BS) void k_bucket_small(const uint32_t* __restrict__ sig, uint32_t n,
                                                     uint32_t* __restrict__ rep) {
  using Sort = rocprim::block_radix_sort<uint32_t, BS, ITEMS, uint32_t>;
  static_assert(sizeof(typename Sort::storage_type) >= 8 * BS, "last items do not fit");
  __shared__ typename Sort::storage_type storage;
  const uint32_t b = blockIdx.x, t = threadIdx.x;
  const uint64_t row = (uint64_t)b * n;
  uint32_t key[ITEMS], val[ITEMS];
  #pragma unroll
  for (int j = 0; j < ITEMS; j++) {
    const uint32_t q = t * ITEMS + j;  // blocked: input order = ascending i
    if (q < n) {
      key[j] = sig_mix(sig[(uint64_t)q * 64 + b]);
      val[j] = q;
      rep[row + q] = q;  // a bucket head keeps its own index
    } else {  // padding sorts after every element (stable)
      key[j] = 0xFFFFFFFFu;
      val[j] = 0xFFFFFFFFu;
    }
  }
  __syncthreads();
  Sort().sort(key, val, storage, 0, 32);
  __syncthreads();  // the storage is free again
  uint32_t* lastk = reinterpret_cast<uint32_t*>(&storage);
  uint32_t* lastv = lastk + BS;
  lastk[t] = key[ITEMS - 1];
  lastv[t] = val[ITEMS - 1];
  __syncthreads();
  uint32_t pk = t ? lastk[t - 1] : 0u, pv = t ? lastv[t - 1] : 0u;
  #pragma unroll
  for (int j = 0; j < ITEMS; j++) {
    const uint32_t q = t * ITEMS + j;
    if (q >= 1 && q < n && key[j] == pk) rep[row + val[j]] = pv;
    pk = key[j];
    pv = val[j];
  }
}

// Past kMapMin records a block takes a band and eight of its partitions, reads
// the band's whole column (64 KiB at most, in L2) through LDS, and each of its
// wavefronts gathers the elements of one partition in index order and passes
// them, 64 at a time, through a table in LDS from value to last index, which is
// each element's predecessor.  A value of kMapOften of the 64 gets registers
// instead, and its elements their predecessors where they are met: through the
// table the wavefront of a value that half of the records share took the block two
// to four times as long.
// A block per band sorting 16 elements a thread leaves three CUs in four idle:
// 8,193 records 71 us against 28 (half of them the same 69 / 32, all 66 / 28), 10,000
// 75 / 27 (72 / 35, 70 / 32), 16,384 97 / 40 (91 / 50, 87 / 44), 200 copies of each 91
// / 68.  At 8,192 the sort's 8 elements a thread take 45, this 34.
// Bound: instructions, every wavefront looking at the whole column, and latency,
// of the LDS round trips of each 64.
constexpr uint32_t kMapSlots = 1024, kMapRing = 512, kMapLoads = 4, kMapWaves = 8;
constexpr int kMapOften = 24;  // of 64: a value that is taken straight from the column
constexpr uint32_t kMapChunk = 4096, kMapPer = kMapChunk / (64 * kMapWaves);
// Partitions of 512 elements or fewer, half the table, and at least a block's.
constexpr uint32_t map_bits(uint32_t n) {
  uint32_t pb = 3;
  while ((n >> pb) > kMapSlots / 2) pb++;
  return pb;
}
__global__ __launch_bounds__(64 * kMapWaves) void k_col_map(const uint32_t* __restrict__ col,
                                                            uint32_t n, uint32_t pb,
                                                            uint32_t* __restrict__ rep) {
  __shared__ uint32_t chunk[kMapChunk];
  __shared__ uint2 rings[kMapWaves][kMapRing];
  __shared__ uint32_t keys[kMapWaves][kMapSlots], lasts[kMapWaves][kMapSlots];
  const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6;
  uint2* const ring = rings[w];
  uint32_t* const key = keys[w];    // 0: free, else the value without its top pb bits, bit 0 set
  uint32_t* const last = lasts[w];  // 0, else the last index of the key's value, plus one
  uint32_t band, at;
  band_block((1u << pb) / kMapWaves, &band, &at);
  at = at * kMapWaves + w;
  const uint32_t* const c = col + (uint64_t)band * n;
  uint32_t* const row = rep + (uint64_t)band * n;
  auto mine = [&](uint32_t h) { return h >> (32 - pb) == at; };
  for (uint32_t k = lane; k < kMapSlots; k += 64) key[k] = last[k] = 0;
  // One wavefront's LDS accesses keep their order; the fences keep the compiler's.
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  uint32_t got = 0, done = 0, values = 0;  // elements gathered, passed on, distinct; uniform
  bool crowded = false;
  // the frequent value, its slot and its last index plus one (0: none yet)
  uint32_t hot = 0, hot_slot = 0, hot_last = 0;
  uint32_t next[kMapPer];
  #pragma unroll
  for (uint32_t k = 0; k < kMapPer; k++) {
    const uint32_t i = 64 * kMapWaves * k + t;
    next[k] = c[i < n ? i : n - 1];
  }
  // The column's elements [q0, stop), which lie in the chunk.  kHot: the frequent
  // value's rows are written here; without one the loop ends after the round that
  // finds it, and its place is returned.
  auto scan = [&](auto has_hot, uint32_t q0, uint32_t stop) {
    constexpr bool kHot = decltype(has_hot)::value;
    for (; q0 < stop; q0 += 64 * kMapLoads) {
      uint32_t h[kMapLoads];
      #pragma unroll
      for (uint32_t k = 0; k < kMapLoads; k++) h[k] = chunk[q0 % kMapChunk + 64 * k + lane];
      if (q0 + 64 * kMapLoads > n) {  // past the column: another partition's
        #pragma unroll
        for (uint32_t k = 0; k < kMapLoads; k++)
          if (q0 + 64 * k + lane >= n) h[k] = (at ^ 1u) << (32 - pb);
      }
      bool quiet = true;  // without the frequent value
      if (kHot) {
        #pragma unroll
        for (uint32_t k = 0; k < kMapLoads; k++) {
          const uint64_t m = __builtin_amdgcn_ballot_w64(h[k] == hot);
          if (!m) continue;
          const uint64_t lower = m & ((1ull << lane) - 1ull);
          const uint32_t prev = lower ? q0 + 64 * k + 63 - __clzll(lower) : hot_last - 1;
          if (__builtin_amdgcn_inverse_ballot_w64(m)) {
            row[q0 + 64 * k + lane] = prev;
            h[k] = (at ^ 1u) << (32 - pb);
          }
          hot_last = q0 + 64 * k + 64 - __clzll(m);
          quiet = false;
        }
      }
      #pragma unroll
      for (uint32_t k = 0; k < kMapLoads; k++) {
        const uint64_t m = __builtin_amdgcn_ballot_w64(mine(h[k]));
        const uint32_t place = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                         __builtin_amdgcn_mbcnt_lo((uint32_t)m, got));
        if (__builtin_amdgcn_inverse_ballot_w64(m))
          ring[place % kMapRing] = make_uint2(h[k], q0 + 64 * k + lane);
        got += (uint32_t)__popcll(m);
      }
      if (crowded) done = got;  // what follows is looked up below
      // The last round, and the one that finds a frequent value, empties the ring.
      bool end = q0 + 64 * kMapLoads >= n, found = false;
      uint32_t often = 0, slot_of_it = 0;
      while (got - done >= 64 || (end && got != done)) {
        if (values + 64 > kMapSlots) {
          crowded = true;
          done = got;
          break;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const bool on = done + lane < got;
        const uint2 e = ring[(done + lane) % kMapRing];
        const uint32_t id = (e.x << pb) | 1u, step = e.x >> 12 | 1u;  // an odd step meets every slot
        uint32_t slot = (e.x >> 3) % kMapSlots;
        bool fresh = false, seek = on;
        while (seek) {
          const uint32_t was = atomicCAS(&key[slot], 0u, id);
          fresh = was == 0;
          seek = was != 0 && was != id;
          if (seek) slot = (slot + step) % kMapSlots;
        }
        values += (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(fresh));
        uint32_t prev = 0, now = 0;
        if (on) {
          prev = __hip_atomic_load(&last[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          atomicMax(&last[slot], e.y + 1);
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          now = __hip_atomic_load(&last[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        // a value again further up in the same 64: the lanes of each such value
        // have the element before them among themselves
        uint64_t again = __builtin_amdgcn_ballot_w64(on && now != e.y + 1);
        const int repeats = __popcll(again);
        while (again) {
          const uint32_t s = __builtin_amdgcn_readlane(slot, __ffsll((unsigned long long)again) - 1);
          const uint64_t same = __builtin_amdgcn_ballot_w64(on && slot == s);
          const uint64_t lower = same & ((1ull << lane) - 1ull);
          if (on && slot == s && lower) prev = ring[(done + 63 - __clzll(lower)) % kMapRing].y + 1;
          again &= ~same;
        }
        if (repeats >= kMapOften && quiet) {  // perhaps the value of some lane in the middle
          const uint32_t s = __builtin_amdgcn_readlane(slot, 21);
          if (__popcll(__builtin_amdgcn_ballot_w64(on && slot == s)) >= kMapOften) {
            often = __builtin_amdgcn_readlane(e.x, 21);
            slot_of_it = s;
            end = found = true;
            if (!kHot) stop = 0;
          }
        }
        if (prev) row[e.y] = prev - 1;
        done = got - done > 64 ? done + 64 : got;
      }
      if (found) {
        if (kHot && lane == 0) atomicMax(&last[hot_slot], hot_last);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        hot = often;
        hot_slot = slot_of_it;
        hot_last = __builtin_amdgcn_readfirstlane(
            __hip_atomic_load(&last[hot_slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
      }
    }
    return q0;
  };
  for (uint32_t c0 = 0; c0 < n; c0 += kMapChunk) {
    __syncthreads();  // every wavefront is through the chunk before
    #pragma unroll
    for (uint32_t k = 0; k < kMapPer; k++) {
      const uint32_t i = c0 + kMapChunk + 64 * kMapWaves * k + t;
      chunk[64 * kMapWaves * k + t] = next[k];
      next[k] = c[i < n ? i : n - 1];
    }
    __syncthreads();
    const uint32_t stop = n - c0 < kMapChunk ? n : c0 + kMapChunk;
    uint32_t q0 = c0;
    if (!hot_last) q0 = scan(std::false_type(), q0, stop);
    if (hot_last) scan(std::true_type(), q0, stop);
  }
  // More values than slots: each predecessor looked up in the column.  No
  // signatures of records crowd like that, so this need only be right.
  for (uint32_t i = lane; crowded && i < n; i += 64) {
    const uint32_t x = c[i];
    if (!mine(x)) continue;
    for (uint32_t q = i; q-- > 0;)
      if (c[q] == x) {
        row[i] = q;
        break;
      }
  }
}

size_t bucket_small_bytes(uint32_t n) { return n > kMapMin ? 256ull * n : 0; }

void launch_bucket_small(const uint32_t* sig, uint32_t n, uint32_t* rep, void* scratch,
                         hipStream_t stream) {
  if (n == 0) return;
  if (n > kBucketSmallMax) throw HipError{NGIA_ERR_ARG, "too many records for the small bucketing"};
  if (n <= 2048) {
    hipLaunchKernelGGL((k_bucket_small<256, 8>), dim3(64), dim3(256), 0, stream, sig, n, rep);
  } else if (n <= kMapMin) {
    hipLaunchKernelGGL((k_bucket_small<1024, 8>), dim3(64), dim3(1024), 0, stream, sig, n, rep);
  } else {
    uint32_t* col = (uint32_t*)scratch;
    const uint32_t pb = map_bits(n);
    hipLaunchKernelGGL(k_mix_columns, dim3((n + 63) / 64), dim3(256), 0, stream, sig, n, col, rep);
    hipLaunchKernelGGL(k_col_map, dim3((64u << pb) / kMapWaves), dim3(64 * kMapWaves), 0, stream, col,
                       n, pb, rep);
  }
  NGIA_HIP(hipGetLastError());
}

// ------------------------------------------------ bucketing of few values
// Signatures of four letters repeat: 200,000 16S reads have about 400 values in
// a band, 4,500 records the most frequent.  Then a table of a band's values
// fits LDS, and a record's predecessor is the last record before it with its
// value's slot:
//  1. k_mix_columns;
//  2. k_value_slots: a tile of a band's column through a table in LDS, then its
//     values into the band's table; each record's slot and each slot's last
//     record in the tile;
//  3. k_value_prefix: each slot's last record before each tile;
//  4. k_value_rows: the records of a tile in order, a wavefront for each 1,024
//     with a table of its own, as in k_col_map; a record that is its value's
//     first there takes the last of the wavefronts before, or before the tile.
// More values than a table holds are noticed, and the full sort takes over.
// Bound: LDS round trips, one chain of them for every 64 records of a wavefront.
constexpr uint32_t kValueSlots = 2048, kValueTile = 8192, kValueThreads = 512;
constexpr uint32_t kValueProbes = 64;
constexpr uint32_t kValuePer = kValueTile / kValueThreads;

// The slot of h in a table of ~h (0: free; the last slot is h = all ones'), or
// kValueSlots when it has no room for it.
__device__ inline uint32_t value_slot(uint32_t* table, uint32_t h) {
  if (h == 0xFFFFFFFFu) return kValueSlots - 1;
  uint32_t s = h % (kValueSlots - 1);
  for (uint32_t probe = 0; probe < kValueProbes; probe++) {
    uint32_t was = __hip_atomic_load(&table[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (was == 0) was = atomicCAS(&table[s], 0u, ~h);
    if (was == 0 || was == ~h) return s;
    s = s + 1 == kValueSlots - 1 ? 0 : s + 1;
  }
  return kValueSlots;
}

__global__ __launch_bounds__(kValueThreads) void k_value_slots(const uint32_t* __restrict__ col,
                                                               uint32_t n, uint32_t tiles,
                                                               uint32_t* __restrict__ tables,
                                                               uint32_t* __restrict__ tile_last,
                                                               uint16_t* __restrict__ slots,
                                                               uint32_t* __restrict__ overflow) {
  __shared__ uint32_t table[kValueSlots], last[kValueSlots], over;
  __shared__ uint16_t slot_of[kValueTile], to_band[kValueSlots];
  const uint32_t t = threadIdx.x;
  uint32_t band, tile;
  band_block(tiles, &band, &tile);
  const uint32_t i0 = tile * kValueTile;
  const uint32_t* const c = col + (uint64_t)band * n;
  for (uint32_t s = t; s < kValueSlots; s += kValueThreads) table[s] = last[s] = 0;
  if (t == 0) over = __hip_atomic_load(overflow, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (over) return;  // another tile's: the rows come from elsewhere
  uint32_t h[kValuePer];
  #pragma unroll
  for (uint32_t k = 0; k < kValuePer; k++) {
    const uint32_t i = i0 + k * kValueThreads + t;
    h[k] = c[i < n ? i : n - 1];
  }
  __syncthreads();
  #pragma unroll
  for (uint32_t k = 0; k < kValuePer; k++) {
    const uint32_t i = i0 + k * kValueThreads + t;
    if (i >= n) continue;
    const uint32_t s = value_slot(table, h[k]);
    if (s == kValueSlots) {
      over = 1;
    } else {
      atomicMax(&last[s], i + 1);
      slot_of[k * kValueThreads + t] = (uint16_t)s;
    }
  }
  __syncthreads();
  for (uint32_t s = t; s < kValueSlots && !over; s += kValueThreads) {
    if (!last[s]) continue;
    const uint32_t b = value_slot(tables + band * kValueSlots, s == kValueSlots - 1 ? 0xFFFFFFFFu : ~table[s]);
    if (b == kValueSlots) {
      over = 1;
    } else {
      to_band[s] = (uint16_t)b;
      tile_last[((uint64_t)band * tiles + tile) * kValueSlots + b] = last[s];
    }
  }
  __syncthreads();
  if (over) {
    if (t == 0) atomicOr(overflow, 1u);
    return;
  }
  #pragma unroll
  for (uint32_t k = 0; k < kValuePer; k++) {
    const uint32_t q = k * kValueThreads + t;
    if (i0 + q < n) slots[(uint64_t)band * n + i0 + q] = to_band[slot_of[q]];
  }
}

// tile_last[band][tile][slot] -> the same over the tiles before.
__global__ __launch_bounds__(256) void k_value_prefix(uint32_t tiles, uint32_t* __restrict__ tile_last) {
  uint32_t* p = tile_last + (uint64_t)blockIdx.y * tiles * kValueSlots + blockIdx.x * 256 + threadIdx.x;
  uint32_t run = 0;
  for (uint32_t t0 = 0; t0 < tiles; t0 += 16) {
    uint32_t v[16];
    #pragma unroll
    for (uint32_t k = 0; k < 16; k++) v[k] = t0 + k < tiles ? p[(uint64_t)(t0 + k) * kValueSlots] : 0u;
    #pragma unroll
    for (uint32_t k = 0; k < 16; k++) {
      if (t0 + k >= tiles) break;
      p[(uint64_t)(t0 + k) * kValueSlots] = run;
      run = v[k] ? v[k] : run;  // later tiles hold larger indices
    }
  }
}

__global__ __launch_bounds__(kValueThreads) void k_value_rows(const uint16_t* __restrict__ slots,
                                                              uint32_t n, uint32_t tiles,
                                                              const uint32_t* __restrict__ before,
                                                              const uint32_t* __restrict__ overflow,
                                                              uint32_t* __restrict__ rep) {
  constexpr uint32_t kWaves = kValueThreads / 64, kSpan = kValueTile / kWaves;
  __shared__ uint32_t lasts[kWaves][kValueSlots];  // a wavefront's last record of each slot, plus one
  if (*overflow) return;
  const uint32_t t = threadIdx.x, lane = t & 63u, w = t >> 6;
  uint32_t band, tile;
  band_block(tiles, &band, &tile);
  const uint32_t i0 = tile * kValueTile;
  const uint64_t row = (uint64_t)band * n;
  uint32_t* const last = lasts[w];
  for (uint32_t s = lane; s < kValueSlots; s += 64) last[s] = 0;
  uint32_t slot[kValuePer], prev[kValuePer];
  #pragma unroll
  for (uint32_t r = 0; r < kValuePer; r++) {
    const uint32_t i = i0 + w * kSpan + 64 * r + lane;
    slot[r] = slots[row + (i < n ? i : n - 1)];
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  #pragma unroll
  for (uint32_t r = 0; r < kValuePer; r++) {
    const uint32_t q = w * kSpan + 64 * r + lane;
    const bool on = i0 + q < n;
    uint32_t now = 0;
    prev[r] = 0;
    if (on) {
      prev[r] = __hip_atomic_load(&last[slot[r]], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      atomicMax(&last[slot[r]], q + 1);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      now = __hip_atomic_load(&last[slot[r]], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    uint64_t again = __builtin_amdgcn_ballot_w64(on && now != q + 1);
    while (again) {  // as in k_col_map
      const uint32_t s = __builtin_amdgcn_readlane(slot[r], __ffsll((unsigned long long)again) - 1);
      const uint64_t same = __builtin_amdgcn_ballot_w64(on && slot[r] == s);
      const uint64_t lower = same & ((1ull << lane) - 1ull);
      if (on && slot[r] == s && lower) prev[r] = w * kSpan + 64 * r + 64 - __clzll(lower);
      again &= ~same;
    }
  }
  __syncthreads();
  const uint32_t* const earlier = before + ((uint64_t)band * tiles + tile) * kValueSlots;
  #pragma unroll
  for (uint32_t r = 0; r < kValuePer; r++) {
    const uint32_t i = i0 + w * kSpan + 64 * r + lane;
    if (i >= n) continue;
    uint32_t p = prev[r];
    for (uint32_t v = w; p == 0 && v-- > 0;) p = lasts[v][slot[r]];
    if (p) {
      p += i0;
    } else {
      p = earlier[slot[r]];
    }
    rep[row + i] = p ? p - 1 : i;
  }
}

namespace {
struct BucketLayout {
  bool wide;
  size_t keys_in, keys_out, vals_in, vals_out, temp, temp_bytes, total;
};
// partitioned path: the band-major column of h, the partitions, their cursors,
// and what the chains left
struct PartLayout {
  bool use;
  uint32_t bits;  // partition bits pb
  size_t col, entries, cursor, left, list, total;
};
PartLayout part_layout(uint32_t n, bool force_wide) {
  PartLayout L{};
  L.use = !force_wide && n <= kPartMaxN;
  if (!L.use) return L;
  L.bits = part_bits(n);
  auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
  const size_t parts = (size_t)64 << L.bits;
  L.col = 0;
  L.entries = L.col + al(256ull * n);
  L.cursor = L.entries + al(8 * parts * kPartCap);
  L.left = L.cursor + al(4 * parts);
  L.list = L.left + al(sizeof(PartsLeft));
  L.total = L.list + al(4 * parts);
  return L;
}
// few values: the column, the slots, and, cleared together, the bands' tables,
// the overflow flag and the last records by tile
struct ValueLayout {
  uint32_t tiles;
  size_t col, slots, tables, overflow, tile_last, total;
};
ValueLayout value_layout(uint32_t n) {
  auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
  ValueLayout L{};
  L.tiles = (n + kValueTile - 1) / kValueTile;
  L.slots = al(256ull * n);
  L.tables = L.slots + al(128ull * n);
  L.overflow = L.tables + 4ull * 64 * kValueSlots;
  L.tile_last = L.overflow + 256;
  L.total = L.tile_last + 4ull * 64 * kValueSlots * L.tiles;
  return L;
}
BucketLayout bucket_layout(uint32_t n, bool force_wide) {
  const uint64_t m = (uint64_t)n * 64;
  BucketLayout L;
  L.wide = force_wide || n > kIdxMask;
  const size_t kb = L.wide ? 8 : 4;
  size_t temp_bytes = 0;
  if (L.wide)
    (void)rocprim::radix_sort_pairs(nullptr, temp_bytes, (uint64_t*)nullptr, (uint64_t*)nullptr,
                                    (uint32_t*)nullptr, (uint32_t*)nullptr, (size_t)m, 0, 38);
  else
    (void)rocprim::radix_sort_pairs(nullptr, temp_bytes, (uint32_t*)nullptr, (uint32_t*)nullptr,
                                    (uint32_t*)nullptr, (uint32_t*)nullptr, (size_t)m, 0, 32);
  auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
  L.keys_in = 0;
  L.keys_out = L.keys_in + al(kb * m);
  L.vals_in = L.keys_out + al(kb * m);
  L.vals_out = L.vals_in + al(4 * m);
  L.temp = L.vals_out + al(4 * m);
  L.temp_bytes = temp_bytes;
  L.total = L.temp + al(temp_bytes);
  return L;
}
}  // namespace

size_t bucket_scratch_bytes(uint32_t n, bool force_wide) {
  const size_t sorted = std::max(bucket_layout(n, force_wide).total, part_layout(n, force_wide).total);
  return !force_wide && n <= kPartMaxN ? std::max(sorted, value_layout(n).total) : sorted;
}

size_t bucket_sort_bytes(uint32_t n, bool force_wide) { return bucket_layout(n, force_wide).total; }

namespace {
// The bucketing of few values; returns false when there were too many (rep then
// holds no result).
bool bucket_values(const uint32_t* sig, uint32_t n, uint32_t* rep, char* s, hipStream_t stream,
                   uint32_t* pinned) {
  const ValueLayout L = value_layout(n);
  uint32_t* col = (uint32_t*)(s + L.col);
  uint16_t* slots = (uint16_t*)(s + L.slots);
  uint32_t* tables = (uint32_t*)(s + L.tables);
  uint32_t* overflow = (uint32_t*)(s + L.overflow);
  uint32_t* tile_last = (uint32_t*)(s + L.tile_last);
  fill_u32(tables, 0, (L.total - L.tables) / 4, stream);
  hipLaunchKernelGGL(k_mix_columns, dim3((n + 63) / 64), dim3(256), 0, stream, sig, n, col, rep);
  hipLaunchKernelGGL(k_value_slots, dim3(64 * L.tiles), dim3(kValueThreads), 0, stream, col, n, L.tiles,
                     tables, tile_last, slots, overflow);
  hipLaunchKernelGGL(k_value_prefix, dim3(kValueSlots / 256, 64), dim3(256), 0, stream, L.tiles,
                     tile_last);
  hipLaunchKernelGGL(k_value_rows, dim3(64 * L.tiles), dim3(kValueThreads), 0, stream, slots, n, L.tiles,
                     tile_last, overflow, rep);
  NGIA_HIP(hipGetLastError());
  uint32_t local = 0;
  uint32_t* over = pinned ? pinned : &local;
  NGIA_HIP(hipMemcpyAsync(over, overflow, 4, hipMemcpyDeviceToHost, stream));
  NGIA_HIP(hipStreamSynchronize(stream));
  return *over == 0;
}

// The time of k_part_left for the partitions past their room, a CU each, against the
// full sort's, in us.  Measured: a column's scan 0.4 ns an element, a partition's
// sorts 4.6 ns of its; the sort 173 us for 20,000 records, 350 for 100,000, 2,400 for
// a million.  All records alike 20,000 records 168 us by the one and 204 by the
// other, 50,000 333 and 255; half of them 100,000 records 401 and 415, a tenth of
// a million 1,522 and 2,970.
bool sort_instead(const PartsLeft& left, uint32_t longs, uint32_t n) {
  const double scan = 0.4e-3 * n, sort = 4.6e-3;
  const double one = scan + sort * left.most, all = (longs * scan + sort * left.elements) / 256;
  return 20 + std::max(one, all) > 120 + 2.3e-3 * n;
}

// The partitioned bucketing; returns false when the full sort must or had better
// redo it (rep then holds a partial result).
bool bucket_partitioned(const PartLayout& L, const uint32_t* sig, uint32_t n, uint32_t* rep,
                        char* s, hipStream_t stream, uint32_t* pinned) {
  const uint32_t pb = L.bits, parts = 64u << pb;
  uint32_t* col = (uint32_t*)(s + L.col);
  uint2* entries = (uint2*)(s + L.entries);
  uint32_t* cursor = (uint32_t*)(s + L.cursor);
  PartsLeft* left = (PartsLeft*)(s + L.left);
  uint32_t* list = (uint32_t*)(s + L.list);
  // the cursors and the counts behind them
  fill_u32(cursor, 0, (L.left - L.cursor + sizeof(PartsLeft)) / 4, stream);
  hipLaunchKernelGGL(k_mix_columns, dim3((n + 63) / 64), dim3(256), 0, stream, sig, n, col, rep);
  const uint32_t tiles = (n + kScatterTile - 1) / kScatterTile;
  hipLaunchKernelGGL(k_part_scatter, dim3(64 * tiles), dim3(kScatterThreads), 0, stream, col, n, pb, tiles, cursor,
                     entries);
  hipLaunchKernelGGL(k_part_chain, dim3(parts), dim3(512), 0, stream, entries, cursor, n, pb, rep, left,
                     list);
  NGIA_HIP(hipGetLastError());
  PartsLeft local{};
  PartsLeft* const got = pinned ? (PartsLeft*)pinned : &local;
  NGIA_HIP(hipMemcpyAsync(got, left, sizeof(PartsLeft), hipMemcpyDeviceToHost, stream));
  NGIA_HIP(hipStreamSynchronize(stream));
  uint32_t most = 0, longs = 0;  // of an XCD, and of all
  for (int x = 0; x < 8; x++) {
    most = std::max(most, got->sorts[x] + got->longs[x]);
    longs += got->longs[x];
  }
  if (most == 0) return true;
  if (longs && sort_instead(*got, longs, n)) return false;
  hipLaunchKernelGGL(k_part_few, dim3(8 * std::min(most, kFewBlocks / 8)), dim3(512), 0, stream, left, list,
                     entries, cursor, n, pb, rep);
  hipLaunchKernelGGL(k_part_left, dim3(8 * std::min(most, 128u)), dim3(512), 0, stream, left, list,
                     entries, cursor, col, n, pb, rep);
  NGIA_HIP(hipGetLastError());
  if (longs == 0) return true;
  NGIA_HIP(hipMemcpyAsync(got, left, sizeof(PartsLeft), hipMemcpyDeviceToHost, stream));
  NGIA_HIP(hipStreamSynchronize(stream));
  return got->overflow == 0;
}
}  // namespace

void launch_bucket(const uint32_t* sig, uint32_t n, uint32_t* rep, void* scratch, size_t bytes,
                   hipStream_t stream, bool force_wide, Values values, uint32_t* pinned) {
  if (n == 0) return;
  const BucketLayout L = bucket_layout(n, force_wide);
  if (bytes < L.total) throw HipError{NGIA_ERR_ARG, "bucketing scratch too small"};
  char* s = (char*)scratch;
  const uint64_t m = (uint64_t)n * 64;
  uint32_t* vals_in = (uint32_t*)(s + L.vals_in);
  uint32_t* vals_out = (uint32_t*)(s + L.vals_out);
  size_t tb = L.temp_bytes;
  const PartLayout P = part_layout(n, force_wide);
  if (P.use && values == Values::kTable && value_layout(n).total <= bytes &&
      bucket_values(sig, n, rep, s, stream, pinned)) return;
  if (P.use && values == Values::kMany && P.total <= bytes &&
      bucket_partitioned(P, sig, n, rep, s, stream, pinned))
    return;
  // the full sort (also when a partition overflowed), from the identity rows
  hipLaunchKernelGGL(k_rep_identity, dim3(grid_for(n, 256), 64), dim3(256), 0, stream, n, rep);
  NGIA_HIP(hipGetLastError());
  if (!L.wide) {
    uint32_t* keys_in = (uint32_t*)(s + L.keys_in);
    uint32_t* keys_out = (uint32_t*)(s + L.keys_out);
    hipLaunchKernelGGL(k_bucket_keys, dim3((n + 63) / 64), dim3(256), 0, stream, sig, n, keys_in,
                       vals_in);
    NGIA_HIP(hipGetLastError());
    NGIA_HIP(rocprim::radix_sort_pairs(s + L.temp, tb, keys_in, keys_out, vals_in, vals_out,
                                       (size_t)m, 0, 32, stream));
    hipLaunchKernelGGL(k_bucket_rep, dim3(grid_for(m, 256)), dim3(256), 0, stream, keys_out,
                       vals_out, m, n, rep);
  } else {
    uint64_t* keys_in = (uint64_t*)(s + L.keys_in);
    uint64_t* keys_out = (uint64_t*)(s + L.keys_out);
    hipLaunchKernelGGL(k_bucket_keys_wide, dim3(grid_for(m, 256)), dim3(256), 0, stream, sig, n,
                       keys_in, vals_in);
    NGIA_HIP(hipGetLastError());
    NGIA_HIP(rocprim::radix_sort_pairs(s + L.temp, tb, keys_in, keys_out, vals_in, vals_out,
                                       (size_t)m, 0, 38, stream));
    hipLaunchKernelGGL(k_bucket_rep_wide, dim3(grid_for(m, 256)), dim3(256), 0, stream, keys_out,
                       vals_out, m, n, rep);
  }
  NGIA_HIP(hipGetLastError());
}

}  // namespace ngia
