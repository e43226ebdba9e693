// dev_graph.hpp -- launchers of dev_graph.hip (device pointers, one stream).
#pragma once

#include "dev_common.hpp"

namespace ngia {

// Pair bins: 0 = scored 0 without alignment, 2..kWinMax = k_align_win<W>,
// kBinWave0 + log2(K) = k_align_wave<K>, kBinPlain = the plain kernel,
// kBinSeg16 / kBinSeg32 = k_align_seg<16, 1> / <32, 1> (several pairs per
// wavefront, one word per lane), kBinSeg16x2..x4 = k_align_seg<16, 2..4>
// (four pairs per wavefront, 2-4 words per lane), kBinSeg8x3 / x2 =
// k_align_seg<8, 3 / 2> (eight pairs per wavefront; x2 only for window bins
// the tuning routes there): band windows of
// kWinMax+1 .. 21 words go to kBinSeg8x3, of 22..30 to kBinSeg16x2, of 31
// words to kBinSeg32, of 32..45 to kBinSeg16x3 and of 46..60 to
// kBinSeg16x4.
constexpr int kBinZero = 0;
constexpr int kBinWave0 = kWinMax + 1;  // kWinMax+1 .. +6 for K = 1..32
constexpr int kBinPlain = kBinWave0 + 6;
constexpr int kBinSeg16 = kBinPlain + 1;
constexpr int kBinSeg32 = kBinSeg16 + 1;
constexpr int kBinSeg16x2 = kBinSeg32 + 1;
constexpr int kBinSeg16x3 = kBinSeg16x2 + 1;
constexpr int kBinSeg16x4 = kBinSeg16x3 + 1;
constexpr int kBinSeg8x3 = kBinSeg16x4 + 1;
constexpr int kBinSeg8x2 = kBinSeg8x3 + 1;
// Bins of one lane per pair with the whole window in registers
// (k_align_lanes): windows of kWinMax+1 .. kLaneMax words have a bin per width
// of their own; kWinLds+1 .. kWinMax share the window bin (k_align_win
// aligns those widths of compact alphabets only); 2 .. kWinLds have a second
// bin, where k_bin_offsets moves the few pairs that do not pay for
// k_align_win<W>, a launch per width.
constexpr int kWinLds = 8;
constexpr int kLaneMax = 40;
constexpr int kBinLane0 = kBinSeg8x2 + 1;
constexpr int kBinLow0 = kBinLane0 + kLaneMax - kWinMax;
constexpr int kBins = kBinLow0 + kWinLds - 1;
static_assert(kBins <= 64, "bin masks are 64-bit");
// The bin of a window of W words, 2..kLaneMax, on one lane per pair.
__host__ __device__ constexpr int lane_bin(int W) {
  return W <= kWinLds ? kBinLow0 + W - 2 : W <= kWinMax ? W : kBinLane0 + W - kWinMax - 1;
}
// The window width of bin b, 0 when it is not one of a single width.
constexpr int bin_width(int b) {
  return b >= kBinLow0    ? b - kBinLow0 + 2
         : b >= kBinLane0 ? b - kBinLane0 + kWinMax + 1
         : b <= kWinMax   ? b
                          : 0;
}
// A kBinSeg16x2 or kBinSeg8x3 bin of fewer pairs goes to kBinSeg32, a
// kBinSeg16x3 or x4 bin to k_align_wave<1> (k_bin_offsets; the seg2_min
// argument of bin_pairs, NGIA_SEG2_MIN): on the heavy-tailed set at -i 90 its
// 14-28k long pairs made the step 0.3 ms longer with two words per lane; the
// log-normal set's 0.37M and 2.3M at -i 70 and 50 took 22% and 20% less
// time.
constexpr uint32_t kSeg2MinPairs = 32768;
// One lane per pair is the cheapest form per word and character (about twice
// the segmented kernels' rate) and the slowest for a single pair: 14 ns per word
// and character, while the whole device does 64 x 1,024 such steps in 9 ns.
// Without a tuned table a bin takes it when a pair is short (at most
// kLaneTiles reference tiles on average) or the round's lane work keeps the
// device busy for about 2.5 times what one of the bin's pairs takes: total
// tiles >= kLaneFill x (an average pair's tiles - kLaneTiles).  Measured, the
// graph at kLaneFill 131,072 / 200,000 / 300,000: 10,000 proteins at -i 70 0.29
// / 0.27 / 0.28 ms, 100,000 at -i 70 0.55 / 0.61 / 0.67, 500,000 at -i 70 2.08 /
// 1.57 / 1.67, 300,000 at -i 60 1.50 / 1.29 / 1.36; kLaneTiles 0 / 100 at
// 300,000: 50,000 of 50-1,000 residues at -i 60 0.59 / 0.48.
constexpr uint32_t kLaneTiles = 80;
constexpr uint32_t kLaneFill = 262144;
// With a tuned table, a group of 17-40-word windows routed to several words
// per lane takes one lane per pair from this many pairs on.
constexpr uint32_t kLaneMinPairs = 65536;
// A window bin of 2..kWinLds words with fewer pairs goes to its lane bin.
constexpr uint32_t kLowLanePairs = 16384;
// Window bins of kWinLds+1..kWinMax words that take neither: with at most
// this many pairs among them a wavefront per pair, else the segmented
// kernels.
constexpr uint32_t kWavePairs = 2048;
// At most this many pairs, none of more than 60 words (no tuned table, not a
// compact alphabet): a wavefront each, past kWaveAllMin words, where a lane takes
// no longer (3 words 17 us, 5 words 24, a wavefront 20).  The device runs
// so many at once, and a wavefront ends a pair sooner than anything else.  The
// step with its pairs, other shapes against this: 500 records, 1,561 pairs 239 / 211
// us; 500, 2,172 236 / 210; 1,000, 2,289 252 / 241; 1,000, 4,448 253 / 282.
constexpr uint32_t kWaveAllPairs = 3072;
constexpr int kWaveAllMin = 4;
// The segmented bins and their (lanes per pair, words per lane).
constexpr bool is_seg_bin(int b) { return b >= kBinSeg16 && b <= kBinSeg8x2; }
constexpr int seg_lanes(int b) {
  return b == kBinSeg32 ? 32 : (b == kBinSeg8x3 || b == kBinSeg8x2) ? 8 : 16;
}
constexpr int seg_words(int b) {
  return b == kBinSeg8x3 ? 3 : b == kBinSeg8x2 ? 2 : b >= kBinSeg16x2 ? b - kBinSeg16x2 + 2 : 1;
}

// Shapes a window bin (W = 2..kWinMax) can be aligned with, chosen per bin
// size by the autotuner: one thread per pair (k_align_win<W>), 16 or 32 lanes
// per pair (k_align_seg), a wavefront per pair (k_align_wave<1>), or 8 lanes
// of two words per pair (k_align_seg<8, 2>).
constexpr uint32_t kShapeWindow = NGIA_SHAPE_WINDOW;
constexpr uint32_t kShapeSeg16 = NGIA_SHAPE_SEG16;
constexpr uint32_t kShapeSeg32 = NGIA_SHAPE_SEG32;
constexpr uint32_t kShapeWave = NGIA_SHAPE_WAVE;
constexpr uint32_t kShapeSeg8 = NGIA_SHAPE_SEG8;
constexpr uint32_t kShapes = kShapeSeg8 + 1;
constexpr int kTuneClasses = NGIA_TUNE_CLASSES;
// Window bin W holding c pairs is aligned with shape[W][k], k the last size
// class with class_size[k] <= c (class 0 below class_size[0]).  Under a zeroed
// table the sizes of the bins and of the round decide (k_bin_offsets).
// Groups of 17..60-word windows: lng[g][k] = NGIA_LONG_* for group g
// (17..21, 22..30, 32..45, 46..60 words) in size class k.
constexpr int kLongGroups = NGIA_LONG_GROUPS;
struct RouteTable {
  uint32_t class_size[kTuneClasses];  // class_size[0] == 0: no table
  uint8_t shape[kWinMax + 1][kTuneClasses];
  uint8_t lng[kLongGroups][kTuneClasses];
};
// Size class of a bin of c pairs.
__host__ __device__ inline uint32_t route_class(const RouteTable& rt, uint32_t c) {
  uint32_t k = 0;
  for (uint32_t j = 1; j < (uint32_t)kTuneClasses; j++)
    if (rt.class_size[j] && rt.class_size[j] <= c) k = j;
  return k;
}

// The bin that aligns window bin W's c pairs under the routing table.
__host__ __device__ inline uint32_t route_window_bin(const RouteTable& rt, uint32_t W, uint32_t c) {
  const uint32_t k = route_class(rt, c);
  switch (rt.shape[W][k]) {
    case kShapeSeg16: return W <= 15 ? (uint32_t)kBinSeg16 : (uint32_t)kBinSeg32;
    case kShapeSeg32: return (uint32_t)kBinSeg32;
    case kShapeWave: return (uint32_t)kBinWave0;
    case kShapeSeg8:
      return W <= 14 ? (uint32_t)kBinSeg8x2 : W <= 15 ? (uint32_t)kBinSeg16 : (uint32_t)kBinSeg32;
    default: return W;
  }
}

// The bins (bit b: bin b) that pairs with windows of wlo..whi words, at most
// `pairs` of them and not of a compact alphabet, can be aligned in after any
// routing of k_bin_offsets; for callers that launch the bins' kernels without
// having read the counts.
uint64_t reachable_bins(uint32_t wlo, uint32_t whi, uint64_t pairs, uint32_t kmax,
                        const RouteTable& route, uint32_t lane_fill);

void fill_u32(uint32_t* p, uint32_t v, uint64_t count, hipStream_t s);
uint64_t scan_scratch_words(uint32_t n);
// out[0..n] = exclusive prefix sums of in[0..n), out[n] = total (n >= 1).
void scan_u32(const uint32_t* in, uint32_t n, uint64_t* out, uint64_t* sums, hipStream_t s);

// Plain form, one band: flags/pos sized n (+1), jobs sized 3n.  parent != null
// selects the fast-mode predicate.
void band_jobs(const uint32_t* rep, const uint32_t* len, uint32_t n, float thr,
               const uint32_t* parent, uint32_t* flags, uint64_t* pos, uint64_t* sums,
               uint32_t* jobs, hipStream_t s);
void jobs_to_edges(const uint32_t* jobs, uint32_t count, uint64_t* ekeys, uint32_t* escores,
                   unsigned long long* ecount, hipStream_t s);
void fast_apply(const uint32_t* jobs, uint32_t count, uint32_t* parent, hipStream_t s);

// A round of the batched fast mode: targets without a parent yet, the pairs
// whose representative first appears in the bands of `bands`; valid receives
// every band with a representative; last: no round follows.
struct FastRound {
  uint32_t* parent = nullptr;  // nullptr: not the fast mode
  uint64_t bands = 0;
  uint64_t* valid = nullptr;
  bool last = false;
};
void fast_resolve(uint32_t n, const uint64_t* off, const uint2* pairs, const uint32_t* score,
                  const uint64_t* keep, const FastRound& fast, unsigned long long* total,
                  hipStream_t s);

// Batched form.
// Candidates: the count pass writes cnt[i] (distinct pairs of target i),
// keep[i] (the bands whose representatives are kept) and adds the count with
// duplicates to *total; after cnt is scanned into off, the emit pass writes
// the pairs grouped by target, in target order.  Targets below t0 get none.
// degree, when not null: n words cleared for edge_count.
void pair_count(const uint32_t* rep, const uint32_t* len, uint32_t n, uint32_t t0, uint32_t bands,
                float thr, uint32_t* cnt, uint64_t* keep, uint32_t* degree,
                unsigned long long* total, hipStream_t s, const FastRound& fast = FastRound());
void pair_emit(const uint32_t* rep, uint32_t n, uint32_t bands, const uint64_t* keep,
               const uint64_t* off, uint2* pairs, hipStream_t s);
// bin_pairs: host_cnt, when not null: pinned memory that gets the bin counts.
void bin_pairs(const uint2* pairs, const uint64_t* npairs, const uint32_t* len, float thr,
               uint32_t* bin_of, uint32_t* bin_cnt, uint32_t* bin_off, uint32_t* cursor,
               uint32_t* list, unsigned long long* bin_tiles, uint32_t* score, uint32_t kmax,
               uint32_t* remap, const RouteTable& route, uint32_t seg2_min, uint32_t lane_fill,
               bool compact, uint32_t grid, hipStream_t s, uint32_t* host_cnt = nullptr);
// One lane per pair over the window bins wlo..whi of a width class (0..3:
// 2-8, 9-16, 17-24 and 25-40 words), widest first; bin_off, bin_cnt, queue
// (kQueueWords words a bin; the launch uses that of whi) and tally are
// indexed by bin.  max_pairs bounds the pairs of the launch.
constexpr int kLaneClasses = 4;
constexpr int lane_class(int W) { return W <= 8 ? 0 : W <= 16 ? 1 : W <= 24 ? 2 : 3; }
constexpr int lane_class_min(int cls) { return cls == 0 ? 2 : 8 * cls + 1; }
constexpr int lane_class_max(int cls) { return cls == 3 ? kLaneMax : 8 * cls + 8; }
void launch_align_lanes(int cls, const AlignArgs& a, const uint2* pairs, const uint32_t* list,
                        const uint32_t* bin_off, const uint32_t* bin_cnt, uint32_t* queue,
                        uint32_t* score, unsigned long long* tally, uint32_t wlo, uint32_t whi,
                        uint32_t cus, uint64_t max_pairs, hipStream_t stream);
void plain_bin_jobs(const uint2* pairs, const uint32_t* list, const uint32_t* bin_off,
                    const uint32_t* bin_cnt, uint32_t* jobs, hipStream_t s);
void plain_bin_scores(const uint32_t* list, const uint32_t* bin_off, const uint32_t* bin_cnt,
                      const uint32_t* jobs, uint32_t* score, hipStream_t s);
// count job triplets (rep, tar, score) as pairs, their number to *npairs; scores
// back into the triplets.
void jobs_to_pairs(const uint32_t* jobs, uint32_t count, uint2* pairs, unsigned long long* npairs,
                   hipStream_t s);
void scores_to_jobs(const uint32_t* score, uint32_t count, uint32_t* jobs, hipStream_t s);
void pairs_to_edges(const uint2* pairs, const uint64_t* npairs, const uint32_t* score,
                    uint64_t* ekeys, uint32_t* escores, unsigned long long* ecount, uint32_t grid,
                    hipStream_t s);

// The sorted edge list of distinct pairs without a sort (dev_graph.hip); off =
// prefix sums of degree (scan_u32), keys_in / scores_in what edge_scatter wrote.
// More edges of one u than this: max_degree tells, and nothing is written.
constexpr uint32_t kMaxDegree = 1024;
void edge_count(const uint2* pairs, const uint64_t* npairs, const uint32_t* score, uint32_t* degree,
                uint32_t* slot, unsigned long long* ecount, unsigned long long* max_degree,
                uint32_t grid, hipStream_t s);
void edge_scatter(const uint2* pairs, const uint64_t* npairs, const uint32_t* score,
                  const uint64_t* off, const uint32_t* slot, const unsigned long long* max_degree,
                  uint64_t* keys, uint32_t* scores, uint32_t grid, hipStream_t s);
// What a round's end tells the host, in pinned memory: `words` of its counters and
// its number of pairs (host null: nothing).
struct RoundReport {
  const uint32_t* counters = nullptr;
  uint32_t words = 0;
  const uint64_t* pairs = nullptr;
  uint32_t* host = nullptr;
  uint64_t* host_pairs = nullptr;
};
void edge_rank(const RoundReport& main, const RoundReport& head, const uint64_t* off, uint32_t n,
               const unsigned long long* max_degree, const uint64_t* keys_in,
               const uint32_t* scores_in, uint64_t* keys, uint32_t* scores, uint32_t grid,
               hipStream_t s);

// m edges as (u, v, (float)score / 100) records of three words.
void edge_records(const uint64_t* keys, const uint32_t* scores, uint64_t m, uint32_t* out,
                  hipStream_t s);

// Sort + unique of m raw edges in place (keys/scores); *d_unique = count.
// The keys are u << 32 | v with u, v < n: the sort skips the bits above
// 32 + bits(n - 1).
size_t finalize_scratch_bytes(uint64_t m);
void finalize_edges(uint64_t* keys, uint32_t* scores, uint64_t m, uint32_t n, uint64_t* keys_tmp,
                    uint32_t* scores_tmp, void* temp, size_t temp_bytes,
                    unsigned long long* d_unique, hipStream_t s);

// Sketch over byte codes (dev_sketch.hip).  The walk form, for databases of at
// most four letters beside rare others: sym_code holds the code of letter y
// in bits 4y..; table (walk_table_bytes) is made by launch_walk_table(sym_code).
size_t walk_table_bytes();
void launch_walk_table(uint32_t sym_code, void* table, hipStream_t stream);
void launch_sketch_walk(const uint32_t* packed, const uint64_t* word_off, const uint8_t* codes,
                        const uint64_t* code_off, const uint32_t* lengths, uint32_t n,
                        uint32_t sym_code, const void* table, uint32_t cus, uint32_t* sig,
                        hipStream_t stream, const uint32_t* list = nullptr);
void launch_sketch(const uint8_t* codes, const uint64_t* code_off, const uint32_t* lengths,
                   uint32_t n, uint32_t* sig, hipStream_t stream, const uint32_t* list = nullptr);
// others[i]: the windows of record i that hold another letter than the four.
void launch_walk_others(const uint32_t* packed, const uint64_t* word_off, const uint32_t* lengths,
                        uint32_t n, uint32_t sym_code, uint32_t* others, hipStream_t stream);
// Whether the walk is a record's shorter way.  Measured, 20 to 28 million
// residues in records of one length, a hash per window against the walk: 500
// bases 254 / 174 us, 400 244 / 326 (many are hashed after all, at fewer
// wavefronts a CU); 1,400 bases with another letter in 4% of the windows 565 / 226,
// 8% 570 / 399, 15% 564 / 727, 82% 567 / 3,701.
constexpr uint32_t kWalkLen = 448;
inline bool walk_fits(uint32_t L, uint32_t others) { return L >= kWalkLen && others <= L / 9; }
// The walk's kernel hashes a record a third slower than k_sketch, whose launch of
// its own lasts as long as its longest record: the records that do not fit get one
// from this share of the residues on.  20,000 records, a few of them hashed: 231 us
// here, 282 in two launches.
constexpr uint32_t kHashRecord = 0x80000000u;
constexpr double kHashShare = 0.1;

}  // namespace ngia
