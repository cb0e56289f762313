// Internal declarations shared by the kernels and the C-ABI layer of libbsx.so.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bsx {

// Extension work is split into bins by query length; each bin runs a kernel
// instantiation.  Index = bin id.  Shape (1, Q) is the two-tasks-per-lane
// kernel (pair.hip, queries of at most Q bases); shape (64, C) the wave kernel
// (wave.hip, queries or bands of at most 64*C columns).  The bins from
// kQueryBins on take the queries of the pair bins where the pair kernel does not
// run them: batches below kPairMinTasks and tasks outside its range (pair_takes).
// Their shape (1, Q) is the task-per-lane kernel (lane.hip), other shapes (L, C) a
// group kernel with L lanes per task and C query columns per lane (qlen <= L*C).
constexpr int kExtBins = 14;
constexpr int kPairBins = 5;
constexpr int kQueryBins = 9;  // bins of the pair and the wave kernels
constexpr int kLaneBins = 2;   // bins of the task-per-lane kernel, after them
struct BinShape { int lanes, cols; };
constexpr BinShape kExtShape[kExtBins] = {{1, 32},  {1, 64},  {1, 96},  {1, 128}, {1, 224}, {64, 4}, {64, 8},
                                          {64, 16}, {64, 32}, {1, 32},  {1, 64},  {16, 6},  {16, 8}, {32, 6}};
constexpr bool is_lane_bin(int b) { return b >= kQueryBins && b < kQueryBins + kLaneBins; }
constexpr int kExtBlock = 64;             // threads per extension block: one wave, so a block
                                          // never holds wave slots idle while a sibling finishes
constexpr int kExtTasksPerBlock = 32;     // four times the task descriptors a plain-kernel block fetches at a time
constexpr int kNarrowTasksPerBlock = 16;  // ... by one narrow-kernel block
constexpr int bin_limit(int b) { return kExtShape[b].lanes * kExtShape[b].cols; }

// The CIGAR (ksw_global2) kernel bins tasks the same way with its own shapes.
constexpr int kGlbBins = 9;
constexpr BinShape kGlbShape[kGlbBins] = {
    {8, 2}, {8, 3}, {8, 4}, {16, 4}, {32, 4}, {64, 4}, {64, 8}, {64, 16}, {64, 32}};
constexpr int kExtSlices = 8;  // slices of a lane kernel's list, each with a fetch counter
// Bins of the two-tasks-per-lane CIGAR kernel (gpair.hip), after the others:
// band widths 2w+1 up to kGlbPairCols, each from glb_pair_top + 1 on.
constexpr int kGlbPairBins = 5;
constexpr int kGlbPairCols[kGlbPairBins] = {15, 23, 31, 47, 63};
__host__ __device__ constexpr int glb_pair_top(int NC) { return NC == 15 ? 0 : NC <= 31 ? NC - 7 : NC - 15; }
constexpr int kGlbAllBins = kGlbBins + kGlbPairBins;
constexpr int kGlbPairTlen = 320;        // longest target of a task of these bins
constexpr int kGlbPairRange = 28000;     // largest size of its scores (16-bit values, -inf = -30000)
// Direction scratch of these bins, a nibble per cell: the share of every bin
// (in 1/64 of the total, kGlbPairScratch bytes per CU) is divided among as many
// waves as have room for 128 tasks of the bin's longest target.  2.5 GB on 256
// CUs; 150 bp reads run 2,000-4,000 waves a bin.
constexpr int64_t kGlbPairScratch = 10 << 20;
constexpr int kGlbPairShare[kGlbPairBins] = {9, 17, 8, 16, 14};
__host__ __device__ constexpr int64_t glb_pair_region(int NC, int rows) { return (int64_t)128 * rows * 4 * ((NC + 7) / 8); }
constexpr int64_t glb_pair_bytes(int num_cu) { return kGlbPairScratch * num_cu; }
// Lists of these bins are ordered by target length, longest first, one bucket
// per length: the tasks of a wave then take equally many rows, and its lanes walk
// back through the same row at the same time (one 768-byte piece of scratch per
// load; with steps of 10 rows the walk fetched a line per lane and took half of
// the kernel's time).  The other bins have one bucket.
constexpr int kGlbKeys = kGlbBins + kGlbPairBins * kGlbPairTlen;
__host__ __device__ constexpr int glb_key(int bin, int tlen) {
  return bin < kGlbBins ? bin : kGlbBins + (bin - kGlbBins) * kGlbPairTlen + (kGlbPairTlen - tlen);
}
// rows of a region for targets of up to tlen bases (whole turns of four rows)
__host__ __device__ constexpr int glb_pair_rows(int tlen) { return (tlen + 3) / 4 * 4; }
// Smallest batch whose narrow bands run the pair kernel: below it the batch
// takes the latency of its waves, and the group kernels finish sooner.  us per
// call, pair / group kernels: 100 bp reads 128,000 tasks 984 / 740, 192,000 1066 /
// 1007, 256,000 1065 / 1291; 150 bp 128,000 1296 / 1097, 160,000 1325 / 1293,
// 192,000 1314 / 1545; 250 bp 100,000 2520 / 1928, 128,000 2478 / 2249, 160,000 2500 /
// 2774.  Tasks of one kind fill the waves sooner: 131,072 of 150 bp reads of half
// band 7 / 15 410 / 721 and 564 / 1096.
constexpr int64_t kGlbPairMinTasks = 131072;
constexpr int glb_bin_limit(int b) { return kGlbShape[b].lanes * kGlbShape[b].cols; }
// First entry of fetch slice s of a list of n entries: a balanced partition,
// the first n % kExtSlices slices hold one entry more.
__host__ __device__ inline uint32_t slice_begin(uint32_t n, int s) {
  const uint32_t q = n / kExtSlices, r = n % kExtSlices;
  return (uint32_t)s * q + ((uint32_t)s < r ? (uint32_t)s : r);
}

// Plain bins list their tasks longest run first, so that a kernel's last
// tasks are short ones and its waves drain together, and so that the tasks of
// one pair-kernel wave, which start together, also end together.  The rows a
// run takes follow min(tlen, 2*h0) closely (the run ends when the target does,
// or once the score built on h0 is spent or the z-drop fires); the key is
// bucketed in steps of 8 rows up to 192 and of 32 beyond, bucket 0 = longest.
// Steps of 32 throughout cost the pair kernels a quarter to a third more rows
// (the waves of a bucket all run as long as its longest run); steps of 4
// changed nothing.  The lists of the lane kernels place rank r of that order at
// slot r / kExtSlices of fetch slice r % kExtSlices, so that every slice is
// itself longest first.  The order changes no result.
constexpr int kRowBuckets = 32;
__host__ __device__ inline int row_bucket(int tlen, int h0) {
  const int est = tlen < 2 * h0 ? tlen : 2 * h0;
  const int k = est < 192 ? (est > 0 ? est >> 3 : 0) : 24 + ((est - 192) >> 5);
  return kRowBuckets - 1 - (k < kRowBuckets - 1 ? k : kRowBuckets - 1);
}

// Learned-band form: classes 0..3 run the band-following frame kernel with
// frames of 24, 40, 80, 144 columns; class 4 is the plain kernel.  Count slots: plain bins
// [0, kExtBins), narrow classes [kExtBins, kExtBins + kBandClasses - 1).
constexpr int kBandClasses = 5;
constexpr int kFrameWidth[kBandClasses - 1] = {24, 40, 80, 144};
constexpr int kCountSlots = 20;
static_assert(kExtBins + kBandClasses - 1 <= kCountSlots, "count slots for bins and narrow classes");
constexpr int kNarrowQMax = 256;  // longest query the narrow kernels take
// Frame classes run by the lane-per-task frame kernel (one task per lane) for
// queries of at most kLaneFrameQMax bases; longer queries of these classes run
// the group frame kernel.  Both compute the same frame run.
constexpr int kLaneFrameClasses = 2;
constexpr int kLaneFrameQMax = 128;
// Fetch counters of an extension call: one for each slice of the lists that the
// task-per-lane kernels take (bins, then frame classes) and one for each group bin,
// each in a line of its own.  A wave of a lane kernel asks every slice of its list
// before it ends, and those atomics on one line wait for one another.  RRBS reads in
// 40-column frames, us per call with a list's counters side by side / so, two runs:
// 98,305 tasks 924, 925 / 887, 924; 300,000 1192, 1204 / 1141, 1176; 1,000,000 1763,
// 1747 / 1710, 1706.  32 words apart measured the same.
constexpr int kFetchPad = 16;  // words from one to the next
constexpr int kLaneLists = kLaneBins + kLaneFrameClasses;
constexpr int lane_fetch(int list) { return list * kExtSlices * kFetchPad; }
constexpr int group_fetch(int bin) { return (kLaneLists * kExtSlices + bin - kQueryBins - kLaneBins) * kFetchPad; }
constexpr int kExtFetchWords = group_fetch(kExtBins);
enum BandMode { kBandPlain = 0, kBandLearned = 1, kBandFixed = 2 };
struct BandPlan {
  int mode;            // BandMode
  int fixed;           // class for kBandFixed
  const uint8_t* cls;  // [n] predicted class for kBandLearned
  bool any_gain;       // route a task to its class even where the frame is not narrower than its bin
  bool skip_plain;     // narrow pass only (labelling): no plain pass, no result unpack
};

// Scores are tracked as (h << 11 | column) keys in 32-bit lanes.
constexpr int kScoreLimit = 1 << 20;
// Largest score of a run of the two-tasks-per-lane kernel of width Q: its
// (score, position) keys and per-column F caps fill 16 bits.
constexpr int pair_score_max(int Q) { return Q <= 128 ? 511 : 255; }
constexpr int kPairMaxTlen = 640;   // with kPairMaxGapExt: the gap cost of a z-drop test,
constexpr int kPairMaxGapExt = 25;  // e * (tlen + Q), and the z-drop itself fit 15 bits
// Smallest binned batch whose short queries run the pair kernel.  A lane runs its
// two tasks serially, so a batch takes at least its longest run (0.4 ms for 100 bp
// reads, 0.8 ms for 150 bp); below this the group kernels, which spread a task
// over 16 lanes, finish sooner.  us per call, pair / group kernels: 100 bp
// 32,000 tasks 429 / 276, 64,000 451 / 431, 128,000 529 / 763; 150 bp 32,000
// 810 / 555, 64,000 874 / 968, 128,000 1406 / 1869.  It decides for timed calls
// only, as others of up to kDirectMaxTasks are not binned; their routing to frame
// classes, which bsx_band_stats counts, goes by these bins too.
constexpr int64_t kPairMinTasks = 65536;

// Kernel-side view of an extension batch (all pointers are device memory).
struct ExtArgs {
  int o_del, e_del, o_ins, e_ins, zdrop, mat_max;
  bool pair;  // the batch's short queries may run the pair kernel
  int qmax;   // no query is longer
  // Query profile by query code qc (0..4): bytes k=0..3 of prof_lo[qc] hold
  // mat[k*5+qc] (target code k), prof_hi[qc] holds mat[20+qc] (target N).
  uint32_t prof_lo[5];
  int32_t prof_hi[5];
  int64_t n;
  const uint8_t* query;
  const uint64_t* q_off;
  const int32_t* qlen;
  const uint8_t* target;
  const uint64_t* t_off;
  const int32_t* tlen;
  const int32_t* h0;
  const int32_t* w;
  const int32_t* end_bonus;
  int32_t *score, *qle, *tle, *gtle, *gscore, *max_off;
  int64_t* cells;
  int32_t* rec_out;  // unbinned batches: [n][8] results as in ExtWork::rec, word 7 = 1 (0: rejected), instead
};

// One task of a bin's work list (written by the binning pass, in bin order).
struct ExtDesc {
  int32_t task, qlen, tlen, h0;
  int32_t w, pad0;  // w already clamped as ksw.c:399-407
  uint32_t qoff_lo, qoff_hi, toff_lo, toff_hi, pad1, pad2;
};
static_assert(sizeof(ExtDesc) == 48, "descriptor layout");

// Side streams of a context: independent launches (the plain bins, the frame
// classes) are spread over the call's stream and these, between a fork and a
// join, so that one launch's tail overlaps the others' work.  All streams keep
// the default priority.
struct StreamSet {
  static constexpr int kSide = 3;
  hipStream_t side[kSide] = {};
  hipEvent_t fork = nullptr, join[kSide] = {};
};
// streams of the plain bins' launches, without and with the pair kernels: 0 =
// the call's stream, k > 0 = side[k-1]
constexpr int kBinStream[2][kExtBins] = {{0, 0, 0, 0, 0, 3, 2, 1, 0, 3, 1, 0, 2, 3},
                                         {0, 3, 2, 1, 0, 3, 2, 1, 3, 2, 1, 3, 1, 2}};
inline hipStream_t pick_stream(const StreamSet* ss, hipStream_t main, int k) {
  return (ss && k > 0 && ss->side[k - 1]) ? ss->side[k - 1] : main;
}
// side streams 1..n wait for the call's stream, and it for them (each costs the
// device a few us of event handling)
inline void ss_fork(const StreamSet* ss, hipStream_t main, int n = StreamSet::kSide) {
  if (!ss || !ss->fork) return;
  (void)hipEventRecord(ss->fork, main);
  for (int k = 0; k < n; ++k) (void)hipStreamWaitEvent(ss->side[k], ss->fork, 0);
}
inline void ss_join(const StreamSet* ss, hipStream_t main, int n = StreamSet::kSide) {
  if (!ss || !ss->fork) return;
  for (int k = 0; k < n; ++k) {
    (void)hipEventRecord(ss->join[k], ss->side[k]);
    (void)hipStreamWaitEvent(main, ss->join[k], 0);
  }
}
// Per-call device workspace for the extension path.
struct ExtWork {
  uint8_t* bin_of;     // [n] bin id, 0xff = rejected task
  ExtDesc* desc;       // [n] task descriptors grouped by bin
  int32_t* rec;        // [n][8] packed per-task results
  uint32_t* counts;    // [kCountSlots] tasks per bin / narrow class
  uint32_t* cursor;    // [kCountSlots] scatter cursors
  uint32_t* fetch;     // [kExtFetchWords] fetch counters (lane_fetch, group_fetch)
  uint32_t* split;     // [2 * kLaneFrameClasses]: per lane-frame class, tasks at the front of its
                       // list (query <= kLaneFrameQMax) and the back-of-list cursor
  int32_t* err;        // [0] rejected count, [1] lowest rejected index
  uint8_t* nbin_of;    // [n] narrow class of the task, 0xff = plain only (learned-band form)
  uint8_t* need_plain; // [n] 1 = the plain kernel computes the task (learned-band form)
  uint32_t* bcount;    // [kExtBins * kRowBuckets] tasks per plain bin and row bucket
  uint32_t* bcursor;   // [kExtBins * kRowBuckets] scatter cursors of the same
  uint32_t* fcount;    // [kLaneFrameClasses * kRowBuckets] front tasks per lane-frame class and row bucket
  uint32_t* fcursor;   // [kLaneFrameClasses * kRowBuckets] scatter cursors of the same
  // optional per-kernel timing: events [2*x], [2*x+1] around timed launch x
  // (time_of_bin, time_of_class, kTimePredict); *tmask gets bit x set for every
  // pair recorded
  hipEvent_t* tev = nullptr;
  uint32_t* tmask = nullptr;
  const StreamSet* ss = nullptr;  // side streams (nullable: everything on the call's stream)
  // tuning: four times the chunk of the plain group kernels, descriptors per block
  // of the frame group kernels, and the shape variant of the bins with alternatives
  int tpb_plain = kExtTasksPerBlock, tpb_narrow = kNarrowTasksPerBlock;
  int shape_var[2] = {0, 0};
};
// The counters of a workspace lie in one array: counts, cursor, err[4], fetch,
// split, bcount, bcursor, fcount, fcursor.
constexpr int kExtCounterWords = 2 * kCountSlots + 4 + kExtFetchWords + 2 * kLaneFrameClasses +
                                 2 * kExtBins * kRowBuckets + 2 * kLaneFrameClasses * kRowBuckets;
inline void ext_counters(ExtWork& wk, uint32_t* p) {
  wk.counts = p;
  wk.cursor = wk.counts + kCountSlots;
  wk.err = (int32_t*)(wk.cursor + kCountSlots);
  wk.fetch = (uint32_t*)(wk.err + 4);
  wk.split = wk.fetch + kExtFetchWords;
  wk.bcount = wk.split + 2 * kLaneFrameClasses;
  wk.bcursor = wk.bcount + kExtBins * kRowBuckets;
  wk.fcount = wk.bcursor + kExtBins * kRowBuckets;
  wk.fcursor = wk.fcount + kLaneFrameClasses * kRowBuckets;
}
// Bins with alternative group shapes (same columns per task, so the binning is
// unchanged; the tuner picks one per device): index 0 = queries of at most 96
// bases, 1 = queries of 97-128.  Variant 0 is kExtShape's shape.
constexpr int kTunedBin[2] = {11, 12};
constexpr BinShape kAltShape[2][2] = {{{16, 6}, {32, 3}}, {{16, 8}, {32, 4}}};
static_assert(kExtShape[kTunedBin[0]].lanes == kAltShape[0][0].lanes &&
              kExtShape[kTunedBin[0]].cols == kAltShape[0][0].cols &&
              kExtShape[kTunedBin[1]].lanes == kAltShape[1][0].lanes &&
              kExtShape[kTunedBin[1]].cols == kAltShape[1][0].cols &&
              kAltShape[0][1].lanes * kAltShape[0][1].cols == bin_limit(kTunedBin[0]) &&
              kAltShape[1][1].lanes * kAltShape[1][1].cols == bin_limit(kTunedBin[1]), "alternative shapes");
// Timed launches: the plain bins, the narrow classes, the predictor.
constexpr int kTimedLaunches = kExtBins + kBandClasses;
constexpr int time_of_bin(int b) { return b; }
constexpr int time_of_class(int c) { return kExtBins + c; }
constexpr int kTimePredict = kTimedLaunches - 1;
static_assert(kTimedLaunches <= 32, "one mask bit per timed launch");
// Slots of bsx_kernel_times, several bins to one where a caller need not tell
// them apart: the query bins, the bins of tasks outside the pair kernel's range
// (those of short queries, then the others), the narrow classes, the predictor.
constexpr int kTimedSlots = 16, kTimedBins = kQueryBins + 2, kOutsideShort = 96;
static_assert(kTimedBins + kBandClasses == kTimedSlots, "timing slots");
constexpr int time_slot(int launch) {
  return launch < kQueryBins ? launch
         : launch < kExtBins ? kQueryBins + (bin_limit(launch) > kOutsideShort ? 1 : 0)
                             : kTimedBins + launch - kExtBins;
}
constexpr int timed_bin_limit(int s) {
  return s < kQueryBins ? bin_limit(s) : s == kQueryBins ? kOutsideShort : bin_limit(kExtBins - 1);
}
inline void time_begin(const ExtWork& wk, int launch, hipStream_t st) {
  if (wk.tev) (void)hipEventRecord(wk.tev[2 * launch], st);
}
inline void time_end(const ExtWork& wk, int launch, hipStream_t st) {
  if (wk.tev) {
    (void)hipEventRecord(wk.tev[2 * launch + 1], st);
    *wk.tmask |= 1u << launch;
  }
}

struct ExtKArgs;
// two-tasks-per-lane kernel of bin `bin` (query width Q), n tasks in the batch
template <int Q>
void launch_pair_bin(const ExtKArgs& k, const ExtWork& wk, int bin, int64_t n, hipStream_t st);
// wave-per-task kernel of bin `bin`, 64 * C columns
template <int C>
void launch_wave_bin(const ExtKArgs& k, const ExtWork& wk, int bin, int64_t n, int num_cu, hipStream_t st);
// Largest batch that runs a wave per task without binning (wave.hip).  us per
// call, so / binned, with pair kernels from 65,536 tasks on: 100 bp reads 500
// tasks 60 / 154, 8,000 97 / 168, 32,000 182 / 278, 80,000 411 / 526, 128,000 703 /
// 565; 150 bp 500 89 / 192, 32,000 278 / 573, 128,000 1044 / 1045; 250 bp 500 192 /
// 330, 80,000 1521 / 2693, 128,000 2925 / 2741.
constexpr int64_t kDirectMaxTasks = 98304;
void launch_direct(const ExtArgs& a, const ExtWork& wk, int num_cu, hipStream_t st, bool cert);
// task-per-lane kernel of bin `bin` (queries of at most Q bases)
template <int Q, bool E1>
void launch_lane_bin(const ExtKArgs& k, const ExtWork& wk, int bin, int64_t n, int num_cu, hipStream_t st, bool pair);
// lane-per-task frame kernel (frame of WF columns) of lane-frame class `cls`
template <int WF, bool E1>
void launch_lane_frame(const ExtKArgs& k, const ExtWork& wk, int cls, int num_cu, hipStream_t st);
hipError_t launch_extend(ExtArgs a, const ExtWork& wk, int num_cu, hipStream_t st, const BandPlan* plan);
// routes a checked batch (nbin_of, need_plain)
void launch_narrow_count(const ExtArgs& a, const ExtWork& wk, int num_cu, hipStream_t st, const BandPlan& plan);
hipError_t launch_narrow(const ExtArgs& a, const ExtKArgs& k, const ExtWork& wk, int num_cu, hipStream_t st,
                         const BandPlan& plan);

struct GlbArgs {
  int o_del, e_del, o_ins, e_ins, mat_max;
  int pen_max;  // largest mat_max - s
  bool pair;    // the batch's narrow bands may run the two-tasks-per-lane kernel
  uint32_t prof_lo[5];
  int32_t prof_hi[5];
  int64_t n;
  const uint8_t* query;
  const uint64_t* q_off;
  const int32_t* qlen;
  const uint8_t* target;
  const uint64_t* t_off;
  const int32_t* tlen;
  const int32_t* w;
  int32_t* score;
  int32_t* n_cigar;
  uint32_t* cigar;
  int64_t cigar_slot;
};

struct GlbWork {
  uint8_t* bin_of;
  int32_t* list;
  uint32_t* counts;
  uint32_t* cursor;
  uint32_t* fetch;
  int32_t* err;  // [0] rejected, [1] first rejected, [2] CIGAR overflows
  uint32_t* kcount;   // [kGlbKeys] tasks per bin and bucket (glb_key)
  uint32_t* kcursor;  // [kGlbKeys] scatter cursors of the same
  uint8_t* z;    // per-group direction-byte slots
  int64_t zslot; // bytes per slot
  uint8_t* zpair;      // direction scratch of the pair kernel (glb_pair_bytes), nullptr without CIGARs or memory
  int64_t pair_bytes;  // this bin's share of it
  const StreamSet* ss;  // side streams for the bins with few tasks per group (nullptr: one stream)
};

constexpr int kGlbMaxT = 1 << 16;
__device__ __forceinline__ int glb_bin_of(int ncol) {
#pragma unroll
  for (int b = 0; b < kGlbBins; ++b)
    if (ncol <= glb_bin_limit(b)) return b;
  return -1;
}
// Whether task t may run: the reference's preconditions, and its directions fit
// a slot.
__device__ __forceinline__ bool glb_task_ok(const GlbArgs& A, const GlbWork& W, int64_t t) {
  const int ql = A.qlen[t], tl = A.tlen[t], w = A.w[t];
  const int diff = tl > ql ? tl - ql : ql - tl;
  const int64_t ncol = ql < 2 * (int64_t)w + 1 ? ql : 2 * (int64_t)w + 1;
  return ql >= 1 && ql <= kGlbMaxT && tl >= 1 && tl <= kGlbMaxT && w >= 0 && glb_bin_of((int)ncol) >= 0 && diff <= w &&
         (A.cigar == nullptr || ncol * tl <= W.zslot);
}
// The bins that take what the unbinned kernel leaves, and the one of a band.
constexpr int kGlbRest = 3;
constexpr int kGlbRestBin[kGlbRest] = {6, 7, 8};
__device__ __forceinline__ int glb_rest_of(int ncol) {
  return ncol <= glb_bin_limit(kGlbRestBin[0]) ? 0 : ncol <= glb_bin_limit(kGlbRestBin[1]) ? 1 : 2;
}
// Largest batch that runs a wave per task without binning (gwave.hip).  us per
// call, so / in bins beside each other: 100 bp reads 300 tasks 55 / 148, 8,000 134 /
// 187, 20,000 252 / 251, 24,000 290 / 266; 150 bp 300 73 / 208, 16,000 298 / 313, 20,000
// 361 / 360, 24,000 416 / 365; 250 bp 300 118 / 308, 16,000 472 / 727, 30,000 794 / 830.
constexpr int64_t kGlbDirectMaxTasks = 20480;
void launch_glb_direct(const GlbArgs& a, const GlbWork& w, hipStream_t st);

// NM / MD:Z / XB:Z of CIGARs (bwa_gen_cigar2's tail, bwa.c:250-343); fields as
// bsx_md_tasks / bsx_md_results in include/bsx.h.
struct MdArgs {
  int64_t n, l_pac, crick_l;
  const uint8_t* opac;
  const int64_t *rb, *re;
  const uint8_t* oquery;
  const uint64_t* oq_off;
  const int32_t* l_query;
  const int32_t* n_cigar;
  const uint32_t* cigar;
  int64_t cigar_slot;
  char* md;
  int64_t md_slot;
  int32_t* md_len;
  char* xb;
  int64_t xb_slot;
  int32_t *xb_len, *nm, *meth, *status;
};
hipError_t launch_md(const MdArgs& a, int num_cu, hipStream_t st);

// SAM CIGAR and position of regions (mem_reg2aln's tail, bwamem.c:1237-1263);
// fields as bsx_reg2aln_tasks / bsx_reg2aln_results in include/bsx.h.
struct Reg2alnArgs {
  int64_t n, l_pac;
  const int64_t *rb, *re;
  const int32_t *qb, *qe, *l_seq, *n_cigar;
  const uint32_t* cigar;
  int64_t cigar_slot;
  uint32_t* out;
  int64_t out_slot;
  int32_t* out_n;
  int64_t* pos;
  int32_t* is_rev;
};
hipError_t launch_reg2aln_cigar(const Reg2alnArgs& a, int num_cu, hipStream_t st);

int64_t glb_groups(int num_cu, bool side);  // scratch slots, with or without the side-stream region
void launch_glb_pair(const GlbArgs& a, const GlbWork& w, int num_cu, hipStream_t st);
// Copies the results of n tasks into pinned memory: rec[n][4] = score, n_cigar,
// first word of the CIGAR in `words` (-1: not there), 1 (0: rejected).  At most
// 2^20 tasks a call.
hipError_t launch_glb_gather(const int32_t* score, const int32_t* n_cigar, const uint32_t* cigar, const uint8_t* bin_of,
                             int n, int64_t slot, int32_t* rec, uint32_t* words, uint32_t room, uint32_t* used,
                             bool clear, hipStream_t st);
constexpr int kGlbGatherWord = kCountSlots;  // its counter, cleared with the call's: cursor[0]
hipError_t launch_global_impl(GlbArgs a, GlbWork w, int num_cu, hipStream_t st);
// counters of a CIGAR call: counts, cursor, err[4], fetch (one a bin), kcount, kcursor
constexpr int kGlbCounterWords = 3 * kCountSlots + 4 + 2 * kGlbKeys;

}  // namespace bsx
