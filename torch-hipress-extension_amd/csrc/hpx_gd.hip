// GradDrop ("DGC") sparsifier: residual accumulation, sampled threshold,
// order-preserving compaction, optional cut to the k largest, scatter decode.
//
// Semantics follow gd_body.h:102-232 (encode) and :283-353 (decode).  The
// reference makes a pass for R += G, a gather for the sample, a full sort of
// the sample, a two-pass copy_if and waits for the stream three times, tensor
// after tensor.  Here every phase is ONE launch for all tensors of a call (a
// table of tensors in the kernel arguments, as in the TBQ and TernGrad paths):
//
//   pick        for samples of up to 65536: the exact threshold by one workgroup per
//               tensor (which gathers small samples itself), in place of select
//   sample      |G[i]+R[i]| at the reference's LCG index stream, gathered
//               BEFORE the update (the same fp32 sum the update will store)
//   select      exact k-th largest of the sample by three radix-histogram
//               passes over the fp32 bit pattern (11+11+10 bits); no sort
//   presample, prepick   in place of these for tensors with large samples: a provisional threshold;
//               behind the pass invert, exact and recount put the exact one in its place
//   stream      ONE pass over the tensor: r = g + r, store r, compare with the
//               threshold, wave64 ballot -> one 64-bit word per 64 elements
//               (bit i = element i), a popcount and the largest |r| per workgroup, and the
//               candidates with their values in a short list per wave
//   finish      tensors that keep up to 2560 entries: one workgroup lists the candidates, cuts
//               them if they are too many and writes the message; the residual is cleared by the pass
//               where it lists a candidate (what a cut drops goes back), else here
//   scan        larger tensors of more than 4096 workgroups, but for those above: exclusive prefix of the
//               per-workgroup counts within chunks of 4096, the chunks' totals and largest |r|
//   expand      larger tensors: folds the totals (each workgroup for itself), reports count,
//               threshold and largest |r| of each tensor to the host; lists (or bit words,
//               where a list was too short) -> ascending indices at their offsets, values out,
//               residual entries zeroed, header written
//
// The stream pass moves 12 bytes per element (g, r in; r out) plus 1/8 byte of
// mask and 8 bytes per candidate; everything else touches O(sample + selected) data.  For tensors
// that keep fewer than 8192 entries that is all: their cut is the device's own business.  For the others the host learns the
// candidate counts from pinned memory while the expand launch is still running
// (it polls the words the expand launch writes first; no wait for the stream), and only
// for tensors with more than `expected` candidates queues the cut, largest |r| first, ties in
// ascending index: one launch of many workgroups, each with a window of the keys, or beyond
// what that is good for (windows_pay) a stable LSD radix sort over as many byte digits as the
// largest key has, whose last pass writes the message.  The expand launch has
// by then left the candidates and their keys where both want them.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <type_traits>
#include <unordered_map>
#include <vector>

#include <immintrin.h>

#include "hpx_common.h"

namespace {
using namespace hpx;

constexpr int kThreads = 256;
constexpr int kPerLane = 16;
constexpr int kTile = kThreads * kPerLane;       // 4096 elements per workgroup
constexpr int kWaveTile = kWave * kPerLane;      // 1024 elements per wave
constexpr int kSelThreads = 1024;
constexpr int kSelBlocksMax = 128;               // few blocks: their bins meet in global atomics
constexpr int kBins1 = 2048, kBins2 = 2048, kBins3 = 1024;  // key = d1:11 | d2:11 | d3:10
constexpr int kHistWords = kBins1 + kBins2 + kBins3;
constexpr int kCapLarge = 256;                   // tensors per launch table (17 KiB of kernel arguments)
constexpr int kCapSmall = 4;                     // calls with a few tensors pass a table of a few hundred bytes

struct alignas(16) GdState {
  uint32_t thr_bits;  // threshold as fp32 bits (provisional path: the provisional one until the exact one is known)
  uint32_t fallback;  // provisional path: 1 when the provisional threshold turned out to lie above the exact one
  uint32_t crowded;   // ... 1 when a wave of the pass found more candidates than its list has room for
  uint32_t ties;      // ... and 1 when the provisional threshold is a value that many samples share
  uint32_t total;     // candidates of a tensor whose cut follows on the device, left by the expand launch
  uint32_t pad[59];
};
constexpr int kHitWays = 128;             // parts of the list of samples above the provisional threshold ...
constexpr uint32_t kWayStep = 32;         // ... whose counters lie in lines of their own, this many words apart
constexpr int64_t kProvisionalAuto = -2;  // the option that leaves the choice to provisional_pays
constexpr int kBySpread = 1 << 20;        // the margin where the caller gives none (see pre_samples)
constexpr uint32_t kPreExpected = 32;     // how many of the samples the provisional threshold is taken from are expected above the exact one
constexpr uint32_t kPreLeast = 32768;     // ... of at least this many samples
constexpr uint32_t kFallback = 0xFFFFFFFEu;  // reported in place of a count: this tensor has to take the other path
constexpr int kScanChunk = 4096;   // per-tile counts scanned by one workgroup
constexpr int kMaxChunks = 128;    // 2^31 elements / kTile / kScanChunk
constexpr int kGroupTiles = 16;    // tiles whose candidates one workgroup of the recount and the expand launch looks after
constexpr uint32_t kPickGather = 1536;   // a sample up to this size is gathered by the one workgroup that takes its threshold
constexpr uint32_t kPickGatherBeside = 256;  // ... where the call has larger ones, and with them a gather launch, anyway
constexpr uint32_t kPickMax = 65536;     // ... and up to this size its threshold is taken by one workgroup
constexpr uint32_t kCutKeep = 8192;      // tensors that keep fewer entries than this are cut on the device ...
constexpr uint32_t kCutLds = 16384;      // ... by one workgroup, which sorts up to this many candidates in LDS: a threshold taken
                                         // from the 80th largest of a sample lets a tenth more or less through

__host__ __device__ constexpr size_t align256(size_t x) { return (x + 255) & ~size_t(255); }
__host__ __device__ constexpr uint32_t cdiv(uint64_t a, uint64_t b) { return static_cast<uint32_t>((a + b - 1) / b); }

constexpr uint32_t kHitExtra = 256 * 128;
// Where the pieces of one tensor's workspace block lie (the same arithmetic on the host and in the kernels).
struct GdLayout {
  size_t state, hist, samples, hitlist, masks, coarse, cnt, wcnt, mx, off, ctot, cmax, end;
};
__host__ __device__ inline GdLayout gd_layout(uint32_t n, uint32_t sample_cnt) {
  const size_t ntiles = cdiv(n, kTile);
  GdLayout l;
  size_t at = 0;
  l.state = at;   at += align256(sizeof(GdState));
  l.hist = at;    at += align256(sizeof(uint32_t) * kHistWords);
  l.samples = at; at += align256(sizeof(uint32_t) * size_t(sample_cnt));
  l.hitlist = at; at += align256(sizeof(uint32_t) * (size_t(sample_cnt) + size_t(kHitExtra)));  // provisional path, see hit_way_room; the finish
  l.masks = at;   at += align256(sizeof(uint64_t) * ntiles * kWave);      // one bit per element
  l.coarse = at;  at += align256(sizeof(uint64_t) * ntiles);              // one bit per mask word: whether it has a bit set
  l.cnt = at;     at += align256(sizeof(uint32_t) * ntiles);              // candidates per tile
  l.wcnt = at;    at += align256(sizeof(uint64_t) * ntiles);              // candidates per wave of a tile, 16 bits each
  l.mx = at;      at += align256(sizeof(uint32_t) * ntiles);              // largest |r| per tile, as bits
  l.off = at;     at += align256(sizeof(uint32_t) * ntiles);              // exclusive prefix within the chunk
  const size_t totals = cdiv(ntiles, kGroupTiles) > uint32_t(kMaxChunks) ? cdiv(ntiles, kGroupTiles) : size_t(kMaxChunks);
  l.ctot = at;    at += align256(sizeof(uint32_t) * totals);              // candidates per chunk, on the provisional path per group
  l.cmax = at;    at += align256(sizeof(uint32_t) * totals);              // largest |r| likewise
  l.end = at;
  return l;
}
// Behind that block: the candidates themselves, (index, value) in ascending order, a list per wave of the pass with room
// for this many (0: no lists, the candidates are looked up through the masks).  Twice the expected number and fourteen: a wave's
// 1024 elements exceed that next to never unless the large ones crowd together, and then the masks name the others.  The pass pays
// for them (138 M elements 229 -> 232 us, ResNet-50's 161 tensors 46.7 -> 48.4, one of a million 4.3 -> 5.1); behind it the
// expand launch takes 9.0 us instead of 14.4 (138 M), and the finish took 8.8 instead of 11.7 for the million, 16.2 instead of 24.8 for
// ResNet-50's 161 (6.1 and 10.3 since).  Up to 12 in 1024: denser, the lists would be a tenth of the tensor.
// Of the tensors that one workgroup settles (gd_finish_kernel) those with few candidates to a list have none either: the masks are
// as quick there, or quicker, and the pass is without the lists' code and stores.  us per encode and decode of one tensor,
// lists / masks: 20 thousand elements, 20 kept 23.3 / 21.7; 80 thousand, 80 kept 25.2 / 23.6; 120 thousand, 120 kept 28.2 / 27.7;
// 32 thousand, 320 kept 25.8 / 24.9; 400 thousand, 400 kept 30.8 / 30.8; 50 thousand, 500 kept 27.1 / 26.9; 80 thousand, 800 kept
// 28.6 / 29.0; 1 M, 1049 kept 32.7 / 34.9; 4 M, 400, 700 and 1200 kept 38.1 / 37.6, 39.3 / 39.4 and 41.4 / 42.9; 8 M, 700, 1200 and 2400
// kept 61.9 / 60.6, 63.5 / 63.6 and 67.1 / 70.7; 16 M, 400 and 2400 kept 87.1 / 77.5 and 93.9 / 89.2; 30 tensors of 150 thousand elements
// together, one in a hundred kept, 31.9 / 30.0.
constexpr uint32_t kFinishKeep = 2560;         // what one workgroup settles: entries kept ...
constexpr uint32_t kFinishTiles = kScanChunk;  // ... and tiles
constexpr uint32_t kListFrom = 400;            // with lists from so many kept ...
constexpr uint32_t kListShare = 6;             // ... and one for so many lists
__host__ __device__ inline bool one_workgroup(uint32_t n, uint32_t limit) { return limit <= kFinishKeep && cdiv(n, kTile) <= kFinishTiles; }
__host__ __device__ inline uint32_t list_room(uint32_t n, uint32_t limit) {
  if (one_workgroup(n, limit) && (limit < kListFrom || limit * (kListShare * uint32_t(kWaveTile)) < n)) return 0;
  const float mean = float(kWaveTile) * float(limit) / float(n);
  return mean > 12.0f ? 0u : (uint32_t(2.0f * mean) + 21u) & ~7u;
}
// Whether the pass leaves zeros in the residual where it lists a candidate's value.  Of a tensor that one workgroup settles nearly all
// candidates are kept, and that workgroup wrote to as many lines of r, at about 700 a microsecond for one CU (ResNet-50's 161
// tensors 16.2 us for that launch, 14.5 with this and the message written in order, the pass as long as before); it puts back
// the few that a cut drops, and all of them where it cannot take them from the lists (gd_finish_kernel).
__host__ __device__ inline bool clears_listed(uint32_t n, uint32_t limit) { return one_workgroup(n, limit) && list_room(n, limit) != 0; }
__host__ __device__ inline size_t list_bytes(uint32_t n, uint32_t limit) {
  return align256(sizeof(uint64_t) * size_t(cdiv(n, kTile)) * (kThreads / kWave) * list_room(n, limit));
}
// The launches behind the pass read them four lanes to a list, so that a wave has the lists of four tiles; the first entries,
// whether there are as many or not, and the lengths are requested together.
constexpr uint32_t kListTiles = 4, kListAhead = 2;
constexpr uint32_t kListLanes = kWave / (kListTiles * (kThreads / kWave));
static_assert(kListLanes * kListTiles * (kThreads / kWave) == kWave && kListAhead * kListLanes <= 16,
              "lanes to a list, and entries a list has room for");
// The cut path's buffers for up to `pairs` candidates: two copies of keys and indices, and the sort's counts.
constexpr int kSortThreads = 1024;
constexpr int kSortPer = 4;
constexpr int kSortTile = kSortThreads * kSortPer;   // tiles of 4096 pairs (8192: each launch of a pass 3 us longer)
constexpr int kSortWaves = kSortThreads / kWave;
constexpr int kSortBinsMax = 512;                    // bins of the widest digit the sort uses (9 bits)
struct CutLayout {
  size_t ka, kb, ia, ib, sc, end;
};
__host__ __device__ inline CutLayout cut_layout(uint64_t pairs) {
  CutLayout c;
  size_t at = 0;
  c.ka = at; at += align256(sizeof(uint32_t) * size_t(pairs));
  c.kb = at; at += align256(sizeof(uint32_t) * size_t(pairs));
  c.ia = at; at += align256(sizeof(int32_t) * size_t(pairs));
  c.ib = at; at += align256(sizeof(int32_t) * size_t(pairs));
  c.sc = at; at += align256(sizeof(uint32_t) * kSortBinsMax * size_t(cdiv(pairs, kSortTile)));
  c.end = at;
  return c;
}

// One tensor of a call.  64 bytes.
struct GdSeg {
  const float* g;      // the gradient
  float* r;            // the array whose entries are selected and cleared: the residual, or (without one) the gradient
  uint8_t* out;        // the message
  uint8_t* ws;         // this tensor's workspace block (gd_layout)
  uint8_t* cut;        // ... and its cut-path buffers (cut_layout)
  uint32_t n;
  uint32_t sample_cnt;
  uint32_t seed;       // low 32 bits of the 64-bit seed
  uint32_t thr_index;  // rank (descending, 0-based) of the threshold in the sample
  uint32_t limit;      // `expected`: more candidates than this are cut to this many
  uint32_t cap;        // pairs the cut-path buffers hold
};
static_assert(sizeof(GdSeg) == 64, "segment record");
// What the expand launch reports per tensor in pinned host memory.
constexpr int kReportWords = 4;  // count of candidates, threshold bits, bits of the largest |r|, unused
constexpr uint32_t kNotReported = 0xFFFFFFFFu;  // a count is < 2^31; as fp32 bits this is a NaN, which no threshold or |r| is
template <int CAP>
struct GdArgs {
  int32_t nseg;
  int32_t residual;             // 0: the sparsifier without residual (dgc_body.h)
  int32_t margin;               // provisional path: how many times the expected number of entries the provisional
                                // threshold lets through, or kBySpread; negative: the gather path
  uint32_t gather;              // the pick launch gathers samples of up to this size itself
  uint32_t listed;              // the tensor's `limit` where the segment's own is set to 0 (a second expand launch), else unused
  int32_t device_cut;           // 1: tensors that keep fewer than kCutKeep entries are cut on the device and report nothing
  int32_t tile_start[CAP + 1];  // exclusive prefix of this launch's workgroups per tensor
  GdSeg seg[CAP];
  uint32_t* report;             // pinned host memory, kReportWords per tensor of this table
};
static_assert(sizeof(GdArgs<kCapLarge>) <= 18000, "kernel-argument budget");

__device__ __forceinline__ uint2* seg_list(const GdSeg& sg, const GdLayout& l) { return reinterpret_cast<uint2*>(sg.ws + l.end); }
__device__ __forceinline__ GdState* seg_state(const GdSeg& sg) { return reinterpret_cast<GdState*>(sg.ws); }

// Rank search in a descending cumulative histogram: returns the bin holding
// rank `rank_in` (0-based from the top) and the rank left inside that bin.
template <int BINS>
__device__ __forceinline__ void find_digit(const uint32_t* __restrict__ hist, uint32_t rank_in,
                                           uint32_t& digit, uint32_t& rank_out) {
  constexpr int PER = BINS / kSelThreads;
  static_assert(PER >= 1, "one bin per thread at least");
  constexpr int kWaves = kSelThreads / kWave;
  __shared__ uint32_t s_wave[kWaves];
  __shared__ uint32_t s_res[2];
  const int t = threadIdx.x;
  const uint32_t lane = t & (kWave - 1), wave = t / kWave;
  uint32_t h[PER], sum = 0;
#pragma unroll
  for (int j = 0; j < PER; j++) {
    h[j] = hist[BINS - 1 - (t * PER + j)];
    sum += h[j];
  }
  // Inclusive prefix over the threads in order: within each wave by lane permutes, then the sixteen wave totals
  // (three workgroup barriers in all; a workgroup-wide scan through LDS, ten rounds of two barriers each, was
  // most of the time of the launches that call this).
  const uint32_t incl = wave_prefix_u32(sum);
  if (lane == kWave - 1) s_wave[wave] = incl;
  if (t == 0) { s_res[0] = 0; s_res[1] = 0; }
  __syncthreads();
  uint32_t before = 0;
#pragma unroll
  for (int w = 0; w < kWaves; w++) before += uint32_t(w) < wave ? s_wave[w] : 0u;
  const uint32_t excl = before + incl - sum;
  if (rank_in >= excl && rank_in - excl < sum) {
    uint32_t c = excl;
#pragma unroll
    for (int j = 0; j < PER; j++) {
      if (rank_in >= c && rank_in - c < h[j]) {
        s_res[0] = uint32_t(BINS - 1 - (t * PER + j));
        s_res[1] = rank_in - c;
      }
      c += h[j];
    }
  }
  __syncthreads();
  digit = s_res[0];
  rank_out = s_res[1];
  __syncthreads();
}

// generate_sample_G, gd_body.h:36-41: naive_int_random<uint32_t>(0, N-1) seeded
// with (uint32)(t + x), one discarded draw, then rand() % N.
__device__ __forceinline__ uint32_t sample_index(uint32_t seed, uint32_t x, uint32_t n) {
  return (lcg_mul(2) * (seed + x) + lcg_add(2)) % n;
}

// One sample per lane: all the random gathers of the sample are in flight at
// once.  The same launch clears the histograms of this call.
template <int CAP>
__global__ __launch_bounds__(kThreads) void gd_sample_kernel(const GdArgs<CAP> a) {
  const int tile = blockIdx.x;
  const int s = find_segment<CAP>(a.tile_start, a.nseg, tile);
  const GdSeg& sg = a.seg[s];
  const GdLayout l = gd_layout(sg.n, sg.sample_cnt);
  uint32_t* hist = reinterpret_cast<uint32_t*>(sg.ws + l.hist);
  uint32_t* samples = reinterpret_cast<uint32_t*>(sg.ws + l.samples);
  const uint32_t x = uint32_t(tile - a.tile_start[s]) * kThreads + threadIdx.x;
  if (x < uint32_t(kHistWords)) hist[x] = 0;
  if (x < sg.sample_cnt) {
    const uint32_t i = sample_index(sg.seed, x, sg.n);
    // with a residual: |G[i] + R[i]|, the value the update is about to store; without (dgc_body.h:18-30): |G[i]|
    samples[x] = __float_as_uint(__builtin_fabsf(a.residual ? sg.g[i] + sg.r[i] : sg.g[i]));
  }
}

template <int PASS>
__device__ __forceinline__ void hist_accumulate(const uint32_t* __restrict__ samples, uint32_t sample_cnt, uint32_t block,
                                                uint32_t nblocks, uint32_t* s_hist, uint32_t prefix) {
  // PASS 1: all keys, digit = key >> 21.  PASS 2: keys with key>>21 == prefix,
  // digit = (key >> 10) & 2047.  PASS 3: keys with key>>10 == prefix, digit = key & 1023.
  const uint32_t stride = nblocks * kSelThreads;
  for (uint32_t x = block * kSelThreads + threadIdx.x; x < sample_cnt; x += stride) {
    const uint32_t key = samples[x];
    if (PASS == 1) {
      atomicAdd(&s_hist[key >> 21], 1u);
    } else if (PASS == 2) {
      if ((key >> 21) == prefix) atomicAdd(&s_hist[(key >> 10) & 2047u], 1u);
    } else {
      if ((key >> 10) == prefix) atomicAdd(&s_hist[key & 1023u], 1u);
    }
  }
}

template <int PASS, int CAP>
__global__ __launch_bounds__(kSelThreads) void gd_select_kernel(const GdArgs<CAP> a) {
  constexpr int BINS = PASS == 1 ? kBins1 : PASS == 2 ? kBins2 : kBins3;
  __shared__ uint32_t s_hist[BINS];
  const int tile = blockIdx.x;
  const int s = find_segment<CAP>(a.tile_start, a.nseg, tile);
  const GdSeg& sg = a.seg[s];
  const GdLayout l = gd_layout(sg.n, sg.sample_cnt);
  uint32_t* hist = reinterpret_cast<uint32_t*>(sg.ws + l.hist);
  for (int i = threadIdx.x; i < BINS; i += kSelThreads) s_hist[i] = 0;
  uint32_t prefix = 0;
  if (PASS >= 2) {
    uint32_t d1, rank;
    find_digit<kBins1>(hist, sg.thr_index, d1, rank);
    prefix = d1;
    if (PASS == 3) {
      uint32_t d2;
      find_digit<kBins2>(hist + kBins1, rank, d2, rank);
      prefix = (d1 << 11) | d2;
    }
  }
  __syncthreads();
  hist_accumulate<PASS>(reinterpret_cast<const uint32_t*>(sg.ws + l.samples), sg.sample_cnt,
                        uint32_t(tile - a.tile_start[s]), uint32_t(a.tile_start[s + 1] - a.tile_start[s]), s_hist, prefix);
  __syncthreads();
  uint32_t* gh = hist + (PASS == 1 ? 0 : PASS == 2 ? kBins1 : kBins1 + kBins2);
  for (int i = threadIdx.x; i < BINS; i += kSelThreads) {
    const uint32_t c = s_hist[i];
    if (c) atomicAdd(&gh[i], c);
  }
}

// One workgroup per tensor.
template <int CAP>
__global__ __launch_bounds__(kSelThreads) void gd_threshold_kernel(const GdArgs<CAP> a) {
  const GdSeg& sg = a.seg[find_segment<CAP>(a.tile_start, a.nseg, blockIdx.x)];
  const GdLayout l = gd_layout(sg.n, sg.sample_cnt);
  const uint32_t* hist = reinterpret_cast<const uint32_t*>(sg.ws + l.hist);
  uint32_t d1, d2, d3, rank;
  find_digit<kBins1>(hist, sg.thr_index, d1, rank);
  find_digit<kBins2>(hist + kBins1, rank, d2, rank);
  find_digit<kBins3>(hist + kBins1 + kBins2, rank, d3, rank);
  if (threadIdx.x == 0) seg_state(sg)->thr_bits = (d1 << 21) | (d2 << 10) | d3;
}

// ---- the sampled threshold without the full gather (provisional path) -----------------------------------------
// The reference's threshold is the thr_index-th largest of a 1 % sample drawn at random positions: gathering it
// costs a 128-byte line of G and one of R per sample, a fifth of the traffic of the pass over the tensor itself,
// and it has to be finished before that pass can start.  This path starts the pass from a PROVISIONAL threshold
// instead - taken from the first samples only (pre_samples) and set low enough that it all but certainly lies below the
// exact one - so the pass lists and marks a superset of the candidates.  Every sample whose value exceeds the
// provisional threshold is then among these, so the exact threshold (the thr_index-th largest of ALL samples) is found
// among the candidates that are samples (gd_invert_kernel).  A last small launch drops the candidates that do not exceed
// the exact threshold; expand goes on as ever.
//
// Values that many elements share (signs, a few levels: gradients that were quantised) may leave the two thresholds equal.  A
// provisional threshold with too many equal samples about it is therefore that value itself, to the last bit (gd_prepick_kernel),
// so that the elements that share it are no candidates, and where so few samples lie above it that it may be the exact one the
// samples equal to it are counted behind the pass (gd_invert_kernel reads all of them, a line of r each): with those above it they
// say that it is.  (Cut off below ten bits as ever it let the sharing elements through, every element of a tensor of signs
// of size 0.0123, or where those bits are zero did not lie below the exact one and the tensor was encoded again.  us per call at 17 M /
// 60 M / 138 M elements: signs of size 0.0123 3494 / 892 / 1130, now 96 / 174 / 340, signs of size 1 170 / 276 / 494, now 97 / 174 / 342;
// through the gather path 142 / 240 / 427.)
//
// Should fewer than thr_index + 1 samples reach the provisional threshold (it lies above the exact one), or should it be a NaN,
// the tensor is reported as kFallback and the host sends it through the gather path, on the residual the pass has already
// updated.
//
// How many samples the provisional threshold is taken from, and its rank among them: as many that kPreExpected of them should lie
// above the exact threshold, and kPreLeast, at a rank eight standard deviations beyond that, so that the exact one lies below the
// provisional one in a case of 10^14.  More samples let less through and take the one workgroup that ranks them longer: 138 M
// elements, a thousandth kept, 16, 32 and 64 expected: 339, 335.4 and 335.4 us a call.  A margin from the caller gives the rank
// in its place, as that many times the number expected.
__host__ __device__ inline uint32_t pre_samples(uint32_t sample_cnt, uint32_t thr_index) {
  uint64_t want = (uint64_t(kPreExpected) * sample_cnt / (uint64_t(thr_index) + 1) + uint64_t(kThreads) - 1) / kThreads * kThreads;
  want = want < kPreLeast ? kPreLeast : want < kPickMax ? want : kPickMax;
  return sample_cnt < want ? sample_cnt : uint32_t(want);
}
__device__ inline uint32_t pre_rank(uint32_t sample_cnt, uint32_t thr_index, int margin, uint32_t s0) {
  uint64_t kp = 0;
  if (margin == kBySpread) {
    const float mean = float(thr_index + 1) * (float(s0) / float(sample_cnt));
    kp = uint64_t(mean + 8.0f * __builtin_sqrtf(mean) + 8.0f);
  } else if (margin > 0) {
    kp = (uint64_t(margin) * (uint64_t(thr_index) + 1) * s0 + sample_cnt - 1) / sample_cnt + 8;
  }
  return kp > s0 - 1 ? s0 - 1 : uint32_t(kp);
}
// How far the number of samples above a threshold strays: four standard deviations, half the provisional threshold's distance.
__device__ inline uint32_t pre_slack(uint32_t sample_cnt, uint32_t thr_index, uint32_t s0) {
  return uint32_t(4.0f * __builtin_sqrtf(float(thr_index + 1) * (float(s0) / float(sample_cnt))) + 4.0f);
}

// Each wave of the launch that gathers the samples leaves its kPreTop largest only.  It holds one key above the
// threshold at most on average (a rank of 490 or so among 32768 samples where one in a hundred is kept); one that holds more
// than it leaves makes the provisional threshold a little lower, which it may be (down to zero where the caller has a tensor
// take this path that keeps one element in ten).
constexpr uint32_t kPreTop = 4;
static_assert(kPickMax / kWave * kPreTop <= 16 * kThreads, "what gd_prepick_kernel holds");

// Rank `rank` (0-based from the top) of `count` keys in global memory, by one workgroup of kSelThreads lanes:
// three histogram passes of 11 + 11 + 10 bits in LDS.  Every lane returns the key.
__device__ __forceinline__ uint32_t select_rank(const uint32_t* __restrict__ keys, uint32_t count, uint32_t rank,
                                                uint32_t* s_hist) {
  uint32_t prefix = 0;
#pragma unroll 1
  for (int pass = 1; pass <= 3; pass++) {
    for (int i = threadIdx.x; i < kBins1; i += kSelThreads) s_hist[i] = 0;
    __syncthreads();
    for (uint32_t x = threadIdx.x; x < count; x += kSelThreads) {
      const uint32_t key = keys[x];
      if (pass == 1) atomicAdd(&s_hist[key >> 21], 1u);
      else if (pass == 2) { if ((key >> 21) == prefix) atomicAdd(&s_hist[(key >> 10) & 2047u], 1u); }
      else if ((key >> 10) == prefix) atomicAdd(&s_hist[key & 1023u], 1u);
    }
    __syncthreads();
    uint32_t d;
    if (pass == 3) find_digit<kBins3>(s_hist, rank, d, rank); else find_digit<kBins1>(s_hist, rank, d, rank);
    prefix = pass == 1 ? d : pass == 2 ? ((prefix << 11) | d) : ((prefix << 10) | d);
  }
  return prefix;
}

// The largest t whose bits below LO are zero and which more than `rank` of the wave's keys (R per lane) reach: with
// LO = 0 the key of that rank (0-based from the top), else a lower bound of it.  Keys are bit patterns of
// non-negative floats, zeros stand for no key; `floor` is a value the key of that rank is known to reach.  One wave, no
// barrier: a bit costs R compares and R counts on the scalar unit, and the bits that the largest key shares with
// the floor cost nothing.
template <int R, int LO>
__device__ __forceinline__ uint32_t wave_rank(const uint32_t (&key)[R], uint32_t rank, uint32_t floor) {
  uint32_t top = 0;
#pragma unroll
  for (int j = 0; j < R; j++) top = key[j] > top ? key[j] : top;
  top = wave_max_u32(top);
  top = __builtin_amdgcn_readfirstlane(top);
  floor = __builtin_amdgcn_readfirstlane(floor);
  const int first = 31 - __builtin_clz((top ^ floor) | 1u);   // bits above it are common to every candidate
  uint32_t t = first < 31 ? (floor >> (first + 1)) << (first + 1) : 0u;
  t = LO > 0 ? (t >> LO) << LO : t;
#pragma unroll 1
  for (int b = first < 30 ? first : 30; b >= LO; b--) {
    const uint32_t c = t | (1u << b);
    uint32_t reach = 0;
#pragma unroll
    for (int j = 0; j < R; j++) reach += uint32_t(__popcll(__ballot(key[j] >= c)));
    if (reach > rank) t = c;
  }
  return t;
}

// The threshold of a tensor whose sample has at most kPickMax entries, by ONE workgroup in one launch; up to kPickGather
// of them it gathers itself (two lines per sample at about 700 random lines a microsecond for one CU: beyond that the
// launch that spreads them over the chip is the quicker one).  The rank wanted is low, a thousandth of the sample, so
// no histogram of the whole sample is needed: of the lanes' largest keys the one of that rank, cut off below its top
// bits, is a lower bound of the threshold that hardly more keys reach than have to; those are listed in LDS (from the three largest that every lane keeps)
// and one wave finds the exact one among them, bit by bit.  Where the bound does not help (a rank beyond the lanes, a
// list that overflows or a lane with more than it keeps: many equal keys) the workgroup takes the three histogram
// passes instead.  The code is kept short on purpose: a launch of one workgroup per tensor meets a cold instruction cache,
// and with the keys in 64 registers and every step unrolled over them this kernel took 9 and 20 us.
// Replaces three histogram launches and a rank search: 1 M elements 15 us in four launches -> 5.2 us in one; ResNet-50's
// 161 tensors 20 -> 7 us, and 4 us less in the gather launch before it.
constexpr uint32_t kPickList = 1024;
constexpr uint32_t kPickAll = 4096;   // listed by a second walk over the sample where the lanes' three largest do not do
// The sum over each row of 16 lanes, in all of its lanes.
__device__ __forceinline__ uint32_t row_sum(uint32_t v) {
  v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x121, 0xF, 0xF, false));   // row_ror:1
  v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x122, 0xF, 0xF, false));
  v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x124, 0xF, 0xF, false));
  v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x128, 0xF, 0xF, false));
  return v;
}
// The sum of a value that repeats every WAVES lanes, by rotations within the rows of 16 lanes.
template <int WAVES>
__device__ __forceinline__ uint32_t sum_of_waves(uint32_t v) {
  static_assert(WAVES == 4 || WAVES == 16, "a power of two, at most a row");
  v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x121, 0xF, 0xF, false));
  v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x122, 0xF, 0xF, false));
  if (WAVES > 4) {
    v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x124, 0xF, 0xF, false));
    v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x128, 0xF, 0xF, false));
  }
  return uint32_t(__builtin_amdgcn_readfirstlane(int(v)));
}
// wave_rank over keys of a whole workgroup of WAVES waves, R a lane: a barrier a bit.  s_part: two rows of a word per wave.
// `stop` is asked before each bit whether the bits so far will do: with how many keys reach what they give (zeros for the rest),
// and how many reach the next such value; on return `above` is the latter.
template <int R, int WAVES, typename Stop>
__device__ __forceinline__ uint32_t workgroup_rank(const uint32_t (&key)[R], uint32_t rank, uint32_t floor, uint32_t (*s_part)[WAVES],
                                                   uint32_t& above, Stop stop) {
  const uint32_t lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  uint32_t top = 0;
#pragma unroll
  for (int j = 0; j < R; j++) top = key[j] > top ? key[j] : top;
  top = wave_max_u32(top);
  if (lane == 0) s_part[0][wave] = top;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < WAVES; w++) top = s_part[0][w] > top ? s_part[0][w] : top;
  top = __builtin_amdgcn_readfirstlane(top);
  floor = __builtin_amdgcn_readfirstlane(floor);
  const int first = 31 - __builtin_clz((top ^ floor) | 1u);   // bits above it are common to every candidate
  uint32_t t = first < 31 ? (floor >> (first + 1)) << (first + 1) : 0u;
  uint32_t least = R * WAVES * kWave;   // keys that reach t
  above = 0;
  int row = 1;
#pragma unroll 1
  for (int b = first < 30 ? first : 30; b >= 0; b--, row ^= 1) {
    if (stop(b, least, above)) break;
    const uint32_t c = t | (1u << b);
    uint32_t reach = 0;
#pragma unroll
    for (int j = 0; j < R; j++) reach += uint32_t(__popcll(__ballot(key[j] >= c)));
    if (lane == 0) s_part[row][wave] = reach;
    __syncthreads();   // the row before it is not written again before everyone is past this one
    reach = sum_of_waves<WAVES>(s_part[row][lane % WAVES]);
    if (reach > rank) { t = c; least = reach; } else above = reach;   // the last that failed is t and one more in the last place
  }
  return t;
}
template <int R, int WAVES = kSelThreads / kWave>
__device__ __forceinline__ uint32_t workgroup_rank(const uint32_t (&key)[R], uint32_t rank, uint32_t floor, uint32_t (*s_part)[WAVES]) {
  uint32_t above;
  return workgroup_rank(key, rank, floor, s_part, above, [](int, uint32_t, uint32_t) { return false; });
}
template <int CAP>
__global__ __launch_bounds__(kSelThreads) void gd_pick_kernel(const GdArgs<CAP> a) {
  __shared__ uint32_t s_hist[kBins1];              // the lanes' largest keys; the histogram of the other way
  __shared__ __align__(16) uint32_t s_list[kPickAll];
  __shared__ uint32_t s_part[2][kSelThreads / kWave];
  __shared__ uint32_t s_n, s_key;
  const GdSeg& sg = a.seg[find_segment<CAP>(a.tile_start, a.nseg, blockIdx.x)];
  const GdLayout l = gd_layout(sg.n, sg.sample_cnt);
  uint32_t* samples = reinterpret_cast<uint32_t*>(sg.ws + l.samples);
  const uint32_t count = sg.sample_cnt, rank = sg.thr_index;
  const uint32_t t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
  auto settle = [&](uint32_t key) { seg_state(sg)->thr_bits = key; };  // one lane
  // the lane's three largest keys
  uint32_t m1 = 0, m2 = 0, m3 = 0;
  auto take = [&](uint32_t k) {
    const uint32_t u = m1 < k ? m1 : k, v = m2 < u ? m2 : u;
    m1 = m1 > k ? m1 : k;
    m2 = m2 > u ? m2 : u;
    m3 = m3 > v ? m3 : v;
  };
  if (count <= a.gather) {
    constexpr int kOwn = (int(kPickGather) + kSelThreads - 1) / kSelThreads;
    float gv[kOwn], rv[kOwn];
#pragma unroll
    for (int j = 0; j < kOwn; j++) {
      const uint32_t x = uint32_t(j) * kSelThreads + t;
      const uint32_t i = x < count ? sample_index(sg.seed, x, sg.n) : 0u;
      gv[j] = x < count ? sg.g[i] : 0.0f;
      rv[j] = x < count && a.residual ? sg.r[i] : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < kOwn; j++) {
      const uint32_t x = uint32_t(j) * kSelThreads + t;
      const uint32_t k = __float_as_uint(__builtin_fabsf(a.residual ? gv[j] + rv[j] : gv[j]));
      if (x < count) samples[x] = k;
      take(k);
    }
  } else {
    // four keys per load, four loads in flight (what lies beyond the sample counts as zero)
    const uint4* __restrict__ quads = reinterpret_cast<const uint4*>(samples);
    const uint32_t last = (count - 1) / 4;
#pragma unroll 1
    for (uint32_t q0 = 0; 4 * q0 < count; q0 += 4 * kSelThreads) {
      uint4 k[4];
#pragma unroll
      for (uint32_t j = 0; j < 4; j++) {
        const uint32_t q = q0 + j * kSelThreads + t;
        k[j] = quads[q < last ? q : last];
      }
#pragma unroll
      for (uint32_t j = 0; j < 4; j++) {
        const uint32_t x = 4 * (q0 + j * kSelThreads + t);
        take(x + 0 < count ? k[j].x : 0u);
        take(x + 1 < count ? k[j].y : 0u);
        take(x + 2 < count ? k[j].z : 0u);
        take(x + 3 < count ? k[j].w : 0u);
      }
    }
  }
  s_hist[t] = m1;
  if (t == 0) s_n = 0;
  __syncthreads();
  // The bound, from the largest keys of groups of lanes: with at least twice as many groups as keys wanted, few groups
  // hide a second one, and a search over 64 keys takes a tenth of the time of one over 1024.  It is cut off at 12
  // mantissa bits (with 4, a sample whose largest values crowd just under one value, as residuals do that are cleared
  // when they pass a threshold, overflowed the list).
  if (wave == 0) {
    constexpr uint32_t kRows = kSelThreads / kWave;
    uint32_t k[kRows];
#pragma unroll
    for (uint32_t j = 0; j < kRows; j++) k[j] = s_hist[j * kWave + lane];
    uint32_t q[4];
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) {
      q[j] = k[j];
#pragma unroll
      for (uint32_t i = j + 4; i < kRows; i += 4) q[j] = k[i] > q[j] ? k[i] : q[j];
    }
    uint32_t one[1] = {q[0]};
#pragma unroll
    for (uint32_t j = 1; j < 4; j++) one[0] = q[j] > one[0] ? q[j] : one[0];
    const uint32_t b = count <= uint32_t(kWave) ? wave_rank<1, 0>(one, rank, 0u)   // the sample itself
                       : rank < 32      ? wave_rank<1, 11>(one, rank, 0u)
                       : rank < 128     ? wave_rank<4, 11>(q, rank, 0u)
                                                : wave_rank<kRows, 11>(k, rank, 0u);
    if (lane == 0) s_key = b;
  }
  __syncthreads();
  const uint32_t bound = s_key;
  if (count <= uint32_t(kWave)) {
    if (t == 0) settle(bound);
    return;
  }
  const bool bounded = rank < uint32_t(kSelThreads) && bound != 0u;   // workgroup-uniform
  // (from 256 keys above the bound on, some lane all but certainly holds four)
  if (bounded && rank < 256u) {
    if (__ballot(m1 >= bound) != 0) {   // most waves hold none
#pragma unroll 1
      for (int j = 0; j < 3; j++) {
        const bool in = m1 >= bound;
        const uint64_t m = __ballot(in);
        if (m == 0) break;
        uint32_t base = 0;
        if (lane == uint32_t(__builtin_ctzll(m))) base = atomicAdd(&s_n, uint32_t(__popcll(m)));
        base = uint32_t(__builtin_amdgcn_readlane(int(base), __builtin_ctzll(m))) + uint32_t(__popcll(m & ((1ull << lane) - 1ull)));
        if (in && base < kPickList) s_list[base] = m1;
        m1 = m2; m2 = m3;
        if (j == 2 && __ballot(in) != 0 && lane == 0) atomicAdd(&s_n, kPickList);   // a lane may hold a fourth: not all are listed
      }
    }
    __syncthreads();
    const uint32_t n = s_n;
    if (n <= kPickList) {
      if (wave == 0) {
        uint32_t found;
        if (n <= kWave) {
          const uint32_t k[1] = {lane < n ? s_list[lane] : 0u};
          found = wave_rank<1, 0>(k, rank, bound);
        } else if (n <= 256) {
          uint32_t k[4];
#pragma unroll
          for (uint32_t j = 0; j < 4; j++) k[j] = j * kWave + lane < n ? s_list[j * kWave + lane] : 0u;
          found = wave_rank<4, 0>(k, rank, bound);
        } else {
          uint32_t k[kPickList / kWave];
#pragma unroll
          for (uint32_t j = 0; j < kPickList / kWave; j++) k[j] = j * kWave + lane < n ? s_list[j * kWave + lane] : 0u;
          found = wave_rank<kPickList / kWave, 0>(k, rank, bound);
        }
        if (lane == 0) settle(found);
      }
      return;
    }
  }
  if (bounded) {
    // Every key from the bound on, by a second walk over the sample (out of the L2).  The histogram passes below would
    // walk it three times, with most keys of a wave in the same few bins: samples of 8000 to 41000 for one entry in a
    // hundred took this launch 35 us, now 23.
    __syncthreads();
    if (t == 0) s_n = 0;
    __syncthreads();
    const uint4* __restrict__ quads = reinterpret_cast<const uint4*>(samples);
    const uint32_t last = (count - 1) / 4;
#pragma unroll 1
    for (uint32_t q0 = 0; 4 * q0 < count; q0 += 4 * kSelThreads) {
      uint4 k[4];
#pragma unroll
      for (uint32_t j = 0; j < 4; j++) {
        const uint32_t q = q0 + j * kSelThreads + t;
        k[j] = quads[q < last ? q : last];
      }
#pragma unroll
      for (uint32_t j = 0; j < 4; j++) {
        const uint32_t x = 4 * (q0 + j * kSelThreads + t);
        const uint32_t v[4] = {k[j].x, k[j].y, k[j].z, k[j].w};
        uint64_t in[4];
        uint32_t all = 0;
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) {
          in[i] = __ballot(x + i < count && v[i] >= bound);
          all += uint32_t(__popcll(in[i]));
        }
        if (all == 0) continue;
        uint32_t base = 0;
        if (lane == 0) base = atomicAdd(&s_n, all);
        base = __builtin_amdgcn_readfirstlane(base);
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) {
          const uint32_t at = base + uint32_t(__popcll(in[i] & ((1ull << lane) - 1ull)));
          if ((in[i] >> lane & 1u) && at < kPickAll) s_list[at] = v[i];
          base += uint32_t(__popcll(in[i]));
        }
      }
    }
    __syncthreads();
    const uint32_t n = s_n;
    if (n <= kPickAll) {
      uint32_t k[4];
#pragma unroll
      for (uint32_t j = 0; j < 4; j++) k[j] = j * kSelThreads + t < n ? s_list[j * kSelThreads + t] : 0u;
      const uint32_t found = workgroup_rank(k, rank, bound, s_part);
      if (t == 0) settle(found);
      return;
    }
  }
  __syncthreads();
  const uint32_t exact = select_rank(samples, count, rank, s_hist);
  if (t == 0) settle(exact);
}

// The first samples, one per lane over many workgroups (one workgroup's gathers into arrays of
// hundreds of megabytes are bound by its CU's address translation: 16384 of them took it 90 us).
template <int CAP>
__global__ __launch_bounds__(kThreads) void gd_presample_kernel(const GdArgs<CAP> a) {
  const int tile = blockIdx.x;
  const int s = find_segment<CAP>(a.tile_start, a.nseg, tile);
  const GdSeg& sg = a.seg[s];
  const GdLayout l = gd_layout(sg.n, sg.sample_cnt);
  uint32_t* samples = reinterpret_cast<uint32_t*>(sg.ws + l.samples);
  const uint32_t s0 = pre_samples(sg.sample_cnt, sg.thr_index);
  const uint32_t x = uint32_t(tile - a.tile_start[s]) * kThreads + threadIdx.x;
  uint32_t key = 0;
  if (x < s0) {
    const uint32_t i = sample_index(sg.seed, x, sg.n);
    key = __float_as_uint(__builtin_fabsf(a.residual ? sg.g[i] + sg.r[i] : sg.g[i]));
  }
  const uint32_t lane = threadIdx.x & (kWave - 1), first = x - lane;
  if (first >= s0) return;
  uint32_t mine = 0;
#pragma unroll
  for (uint32_t j = 0; j < kPreTop; j++) {
    uint32_t top = key;
    top = wave_max_u32(top);
    if (lane == j) mine = top;
    if (lane == uint32_t(__builtin_ctzll(__ballot(key == top)))) key = 0;
  }
  if (lane < kPreTop) samples[first / kWave * kPreTop + lane] = mine;
}

// The provisional threshold from what the waves of that launch have left, by one workgroup of four waves for each tensor: the
// key of the rank wanted, cut off below ten bits of mantissa (a lower threshold will do) unless a crowd of keys shares these,
// too many for all of them to lie above the exact threshold by chance: then to the last bit.  Its code is short because it is
// fetched anew in every call, and a barrier a bit is cheap among four waves: with all samples ranked by gd_pick_kernel this
// launch took 7.3 us, and 13 in two calls of five; by sixteen waves 6.8; now 5.2, and 5.6 since it looks for
// crowds (138 M elements, 32 thousand samples).
template <int CAP>
__global__ __launch_bounds__(kThreads) void gd_prepick_kernel(const GdArgs<CAP> a) {
  __shared__ uint32_t s_part[2][kThreads / kWave];
  const GdSeg& sg = a.seg[blockIdx.x];
  const GdLayout l = gd_layout(sg.n, sg.sample_cnt);
  const uint32_t s0 = pre_samples(sg.sample_cnt, sg.thr_index), rank = pre_rank(sg.sample_cnt, sg.thr_index, a.margin, s0);
  const uint32_t slack = pre_slack(sg.sample_cnt, sg.thr_index, s0);
  const uint32_t quads = cdiv(s0, kWave) * (kPreTop / 4), t = threadIdx.x;
  const uint4* __restrict__ left = reinterpret_cast<const uint4*>(sg.ws + l.samples);
  auto settle = [&](auto rounds) {
    constexpr uint32_t kRounds = decltype(rounds)::value;
    uint32_t key[4 * kRounds];
#pragma unroll
    for (uint32_t j = 0; j < kRounds; j++) {
      const uint4 q = j * kThreads + t < quads ? left[j * kThreads + t] : make_uint4(0, 0, 0, 0);
      key[4 * j] = q.x; key[4 * j + 1] = q.y; key[4 * j + 2] = q.z; key[4 * j + 3] = q.w;
    }
    if (t < uint32_t(kHitWays)) *reinterpret_cast<uint2*>(sg.ws + l.hist + t * kWayStep * sizeof(uint32_t)) = make_uint2(0, 0);
    uint32_t above;
    const uint32_t found = workgroup_rank(key, rank, 0u, s_part, above,
                                          [=](int b, uint32_t least, uint32_t above) { return b == 12 && least - above <= slack; });
    if (t == 0) {
      GdState* st = seg_state(sg);
      st->thr_bits = found;
      st->fallback = found > 0x7F800000u ? 1u : 0u;   // a NaN: every element would be a candidate, and which of them are above it?
      st->crowded = 0;
      // so few samples above it that it may be the exact one; zero need not be counted, nothing lies below it
      st->ties = found != 0 && float(above) < float(sg.thr_index + 1) * (float(s0) / float(sg.sample_cnt)) + float(slack) ? 1u : 0u;
    }
  };
  if (quads <= 2 * kThreads) settle(std::integral_constant<uint32_t, 2>{}); else settle(std::integral_constant<uint32_t, 4>{});
}

// The candidates that are samples, listed with their values, in one of two ways.
//
// Large tensors look no sample up: each of the pass's few candidates works out how often it was
// sampled.  Sample x is element (A (x + seed) + B mod 2^32) mod n, and A is odd: an element i is the sample of the x for
// which that word is one of i, i + n, i + 2 n, ..., and from one of these words to the next x advances by n / A mod
// 2^32.  2^32 / n additions and compares for each candidate, 32 for 138 M elements: for its 360 thousand candidates
// this launch takes 7 us, the look-up of its 1.4 million samples took 13.  Four lanes to a list, as in the expand launch.
//
// Where a list was too short for its candidates (the large values lie together: whole rows of an embedding's gradient),
// and in small tensors, where a candidate's steps are many, every sample is looked up in the bit mask instead.  That is the
// same work wherever the candidates lie.  When a wave walked the masks of such tiles instead, thousands of candidates of 2^32 / n
// steps each, this launch took 782 us for 17 M elements, half of the large ones among them within one element in 1500, and
// 271 for 138 M; now 12 and 14.5.  The whole call: 927 -> 150 and 792 -> 518 us, 150 and 556 through the gather path.
constexpr uint32_t kInverseFrom = 1u << 24;   // elements: 256 steps a candidate
__host__ __device__ constexpr uint32_t odd_inverse(uint32_t a) {
  uint32_t v = a;                             // right to 3 bits; each step doubles them
  for (int i = 0; i < 4; i++) v *= 2 - a * v;
  return v;
}
constexpr uint32_t kLcgInverse = odd_inverse(lcg_mul(2));
static_assert(kLcgInverse * lcg_mul(2) == 1u, "the multiplier has an inverse mod 2^32");
// What is found goes to one of kHitWays parts of a list (one counter for all would take the few thousand appends one after
// the other, 37 ns each): samples 256 b to 256 b + 255 to part b % kHitWays, which has room for all of them, or the candidates of
// workgroup b.
__host__ __device__ inline uint32_t hit_way_room(uint32_t sample_cnt) {
  const uint32_t blocks = cdiv(sample_cnt, kThreads);
  return cdiv(blocks, kHitWays) * uint32_t(kThreads);
}
constexpr int kLook = 4;   // blocks of samples a workgroup looks up together, so that their loads are in flight together
template <int CAP>
__global__ __launch_bounds__(kThreads) void gd_invert_kernel(const GdArgs<CAP> a) {
  const int blk = blockIdx.x;
  const int s = find_segment<CAP>(a.tile_start, a.nseg, blk);
  const GdSeg& sg = a.seg[s];
  const GdLayout l = gd_layout(sg.n, sg.sample_cnt);
  const uint32_t n = sg.n, ntiles = cdiv(n, kTile), lane = threadIdx.x & (kWave - 1);
  const uint4 st = *reinterpret_cast<const uint4*>(seg_state(sg));   // GdState's first four words, uniform
  const uint32_t own = uint32_t(blk - a.tile_start[s]);
  const uint32_t tile0 = (own * (kThreads / kWave) + threadIdx.x / kWave) * kListTiles;
  const uint32_t room = list_room(n, sg.limit), sub = lane % kListLanes, mine = tile0 * (kThreads / kWave) + lane / kListLanes;
  const bool my_tile = tile0 + lane / (kListLanes * (kThreads / kWave)) < ntiles;
  const uint2* __restrict__ list = seg_list(sg, l) + size_t(mine) * room;
  uint2 p[kListAhead];
  uint32_t listed = 0;
  if (n >= kInverseFrom && my_tile) {
    listed = reinterpret_cast<const uint16_t*>(sg.ws + l.wcnt)[mine];
    if (room != 0) {
#pragma unroll
      for (uint32_t q = 0; q < kListAhead; q++) p[q] = list[q * kListLanes + sub];
    }
  }
  const uint32_t way_room = hit_way_room(sg.sample_cnt);
  auto append = [&](uint32_t way, bool hit, uint32_t key) {   // by all lanes
    const uint64_t m = __ballot(hit);
    if (m == 0) return;
    uint32_t base = 0;
    if (lane == uint32_t(__builtin_ctzll(m)))
      base = atomicAdd(reinterpret_cast<uint32_t*>(sg.ws + l.hist) + way * kWayStep, uint32_t(__popcll(m)));
    base = uint32_t(__builtin_amdgcn_readlane(int(base), __builtin_ctzll(m))) + uint32_t(__popcll(m & ((1ull << lane) - 1ull)));
    if (!hit) return;
    if (base < way_room) reinterpret_cast<uint32_t*>(sg.ws + l.hitlist)[size_t(way) * way_room + base] = key;
    else seg_state(sg)->fallback = 1;
  };
  if (st.y) return;   // fallback: a NaN, or noted by a wave before; what is listed will not be used
  const uint32_t blocks = cdiv(sg.sample_cnt, kThreads), groups = uint32_t(a.tile_start[s + 1] - a.tile_start[s]);
  if (st.w) {   // ties
    const uint32_t thr_bits = st.x;
    const float thr = __uint_as_float(thr_bits);
    uint32_t equal = 0;   // the wave's
#pragma unroll 1
    for (uint32_t b = own; b < blocks; b += kLook * groups) {
      float v[kLook];
      bool any[kLook];
#pragma unroll
      for (uint32_t q = 0; q < uint32_t(kLook); q++) {
        const uint64_t x = (uint64_t(b) + uint64_t(q) * groups) * kThreads + threadIdx.x;
        any[q] = x < sg.sample_cnt;
        v[q] = any[q] ? sg.r[sample_index(sg.seed, uint32_t(x), n)] : 0.0f;
      }
#pragma unroll
      for (int q = 0; q < kLook; q++) {
        const uint32_t key = __float_as_uint(v[q]) & 0x7FFFFFFFu;
        equal += uint32_t(__popcll(__ballot(any[q] && key == thr_bits)));
        append((b + uint32_t(q) * groups) % uint32_t(kHitWays), any[q] && !(__builtin_fabsf(v[q]) <= thr), key);
      }
    }
    if (lane == 0 && equal != 0)
      atomicAdd(reinterpret_cast<uint32_t*>(sg.ws + l.hist) + own % uint32_t(kHitWays) * kWayStep + 1, equal);
    return;
  }
  if (n < kInverseFrom || st.z) {   // crowded
    const uint64_t* __restrict__ masks = reinterpret_cast<const uint64_t*>(sg.ws + l.masks);
    const uint64_t* __restrict__ coarse = reinterpret_cast<const uint64_t*>(sg.ws + l.coarse);
#pragma unroll 1
    for (uint32_t b = own; b < blocks; b += kLook * groups) {
      uint32_t i[kLook], key[kLook];
      uint64_t c[kLook], m[kLook];
      bool hit[kLook];
      // first whether the element's mask word has any bit at all (one bit per word: the whole map stays in cache),
      // and only then the word itself, and the value
#pragma unroll
      for (uint32_t q = 0; q < uint32_t(kLook); q++) {
        const uint64_t x = (uint64_t(b) + uint64_t(q) * groups) * kThreads + threadIdx.x;
        hit[q] = x < sg.sample_cnt;
        i[q] = sample_index(sg.seed, uint32_t(x), n);
        c[q] = hit[q] ? coarse[i[q] >> 12] : 0ull;
      }
#pragma unroll
      for (int q = 0; q < kLook; q++) m[q] = (c[q] >> ((i[q] >> 6) & 63u)) & 1ull ? masks[i[q] >> 6] : 0ull;
#pragma unroll
      for (int q = 0; q < kLook; q++) {
        hit[q] = (m[q] >> (i[q] & 63u)) & 1ull;
        key[q] = hit[q] ? __float_as_uint(sg.r[i[q]]) & 0x7FFFFFFFu : 0u;
      }
#pragma unroll
      for (int q = 0; q < kLook; q++) append((b + uint32_t(q) * groups) % uint32_t(kHitWays), hit[q], key[q]);
    }
    return;
  }
  const uint32_t steps = 0xFFFFFFFFu / n, step = kLcgInverse * n, last = 0xFFFFFFFFu - steps * n;
  auto sampled = [&](uint32_t i) {
    uint32_t x = kLcgInverse * (i - lcg_add(2)) - sg.seed, times = 0;
#pragma unroll 4
    for (uint32_t m = 0; m < steps; m++, x += step) times += x < sg.sample_cnt ? 1u : 0u;
    return times + (i <= last && x < sg.sample_cnt ? 1u : 0u);
  };
  auto note = [&](uint32_t times, uint32_t key) {
    for (; __ballot(times != 0) != 0; times -= times != 0 ? 1u : 0u) append(own % uint32_t(kHitWays), times != 0, key);
  };
  uint32_t times[kListAhead];
#pragma unroll
  for (uint32_t q = 0; q < kListAhead; q++) times[q] = q * kListLanes + sub < listed ? sampled(p[q].x) : 0u;
#pragma unroll
  for (uint32_t q = 0; q < kListAhead; q++) note(times[q], p[q].y & 0x7FFFFFFFu);
  for (uint32_t j = kListAhead * kListLanes; __ballot(j < listed) != 0; j += kListLanes) {
    const bool any = j + sub < listed;
    const uint2 e = any ? list[j + sub] : make_uint2(0, 0);
    note(any ? sampled(e.x) : 0u, e.y & 0x7FFFFFFFu);
  }
}

// One workgroup per tensor: the exact threshold from the samples that were found, or the other path called for.  Eight lanes
// take a part of the list, up to R keys each, and the rank is found among the keys in registers (rank_hits); only if a
// part is longer than that are they drawn together (into the samples' block, free by now) and ranked by histograms.
// (Drawn together first, then the bits tried one by one: 12 thousand keys 27 us, 18.5 from the registers.)
constexpr uint32_t kWayLanes = kSelThreads / kHitWays;
// The hits' distances from the provisional threshold go into 2048 bins by exponent and six further bits, larger ones first, as
// a cut's do (cut_bin); the bin that the rank falls into holds a handful, and one wave finds the key among them.  Where it holds
// more than a wave has lanes (few distinct values) the bits are tried one after the other, a barrier a bit.  (That way for
// all, sixteen waves counting: the launch 10.5 us for the 2300 hits of 138 M elements, now 5.4.)
constexpr uint32_t kHitBins = 2048;
template <int R>
__device__ __forceinline__ uint32_t rank_hits(const uint32_t* __restrict__ part, uint32_t count, uint32_t rank, uint32_t floor,
                                              uint32_t (*s_part)[kSelThreads / kWave], uint32_t* s_hist, uint32_t* s_few, uint32_t* s_found) {
  static_assert(kHitBins == uint32_t(kBins1) && kHitBins == 2 * kSelThreads && kSelThreads / kWave == 16, "two bins a lane, a row of waves");
  const uint32_t t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
  auto bin_of = [=](uint32_t key) {   // (held to the bins also for what is no distance)
    const uint32_t bin = kHitBins - 1 - ((__float_as_uint(float(key - floor)) >> 17) - (127u << 6));
    return bin < kHitBins ? bin : kHitBins - 1;
  };
  uint32_t k[R];
#pragma unroll
  for (uint32_t j = 0; j < uint32_t(R); j++) {
    const uint32_t at = j * kWayLanes + threadIdx.x % kWayLanes;
    k[j] = at < count ? part[at] : 0u;   // a hit is above the floor
  }
  reinterpret_cast<uint2*>(s_hist)[t] = make_uint2(0, 0);
  if (t == 0) s_found[2] = 0;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < R; j++)
    if (k[j] != 0) atomicAdd(&s_hist[bin_of(k[j])], 1u);
  __syncthreads();
  const uint2 c = reinterpret_cast<const uint2*>(s_hist)[t];
  const uint32_t incl = wave_prefix_u32(c.x + c.y);
  if (lane == kWave - 1) s_part[0][wave] = incl;
  __syncthreads();
  const uint32_t sum = s_part[0][lane & 15], sums = row_prefix_u32(sum);
  const uint32_t at = uint32_t(__builtin_amdgcn_readlane(int(sums - sum), __builtin_amdgcn_readfirstlane(int(wave)))) + incl - c.x - c.y;
  if (rank >= at && rank - at < c.x + c.y) {   // one lane, there are more than `rank`
    const bool second = rank - at >= c.x;
    s_found[0] = 2 * t + (second ? 1u : 0u);
    s_found[1] = at + (second ? c.x : 0u);
  }
  __syncthreads();
  const uint32_t bin = s_found[0], before = s_found[1];
  if (s_hist[bin] <= uint32_t(kWave)) {   // uniform
#pragma unroll
    for (int j = 0; j < R; j++)
      if (k[j] != 0 && bin_of(k[j]) == bin) s_few[atomicAdd(&s_found[2], 1u)] = k[j];
    __syncthreads();
    const uint32_t few[1] = {lane < s_hist[bin] ? s_few[lane] : 0u};
    return wave == 0 ? wave_rank<1, 0>(few, rank - before, floor) : 0u;   // the first wave's is used
  }
  __syncthreads();   // everyone has read the waves' sums
  return workgroup_rank(k, rank, floor, s_part);
}
template <int CAP>
__global__ __launch_bounds__(kSelThreads) void gd_exact_kernel(const GdArgs<CAP> a) {
  __shared__ __align__(16) uint32_t s_hist[kBins1];
  __shared__ uint32_t s_part[2][kSelThreads / kWave], s_few[kWave], s_found[3];
  __shared__ uint32_t s_off[kHitWays];
  const GdSeg& sg = a.seg[blockIdx.x];
  const GdLayout l = gd_layout(sg.n, sg.sample_cnt);
  GdState* st = seg_state(sg);
  const uint32_t t = threadIdx.x, lane = t & (kWave - 1);
  const uint32_t prov = st->thr_bits, way = t / kWayLanes, room = hit_way_room(sg.sample_cnt);
  const uint32_t* ways = reinterpret_cast<const uint32_t*>(sg.ws + l.hist);
  const uint32_t* parts = reinterpret_cast<const uint32_t*>(sg.ws + l.hitlist);
  static_assert(kHitWays == 2 * kWave && kHitWays * kWayStep <= uint32_t(kHistWords), "two counts a lane, in the histograms' block");
  const uint32_t mine = ways[way * kWayStep];
  const uint32_t c0 = ways[2 * lane * kWayStep], c1 = ways[(2 * lane + 1) * kWayStep];   // every wave for itself
  if (st->fallback) return;   // uniform: not all that were found had room
  const uint32_t incl = wave_prefix_u32(c0 + c1), most = wave_max_u32(c0 > c1 ? c0 : c1);
  const uint32_t found = __builtin_amdgcn_readlane(incl, kWave - 1);
  __syncthreads();   // nobody reads the state below
  if (found <= sg.thr_index) {
    // all other samples are at most the provisional threshold: it is the exact one if enough of them are equal to it (nothing is
    // less than zero, so that one is known)
    uint32_t equal = 0;
    if (st->ties) equal = ways[2 * lane * kWayStep + 1] + ways[(2 * lane + 1) * kWayStep + 1];
    equal = wave_sum_u32(equal);
    if (t == 0 && prov != 0 && found + equal <= sg.thr_index) st->fallback = 1;
    return;
  }
  const uint32_t* part = parts + size_t(way) * room;
  uint32_t key;
  if (most <= 8 * kWayLanes) {
    key = rank_hits<8>(part, mine, sg.thr_index, prov, s_part, s_hist, s_few, s_found);
  } else if (most <= 32 * kWayLanes) {
    key = rank_hits<32>(part, mine, sg.thr_index, prov, s_part, s_hist, s_few, s_found);
  } else {
    if (t < uint32_t(kWave)) { s_off[2 * lane] = incl - c0 - c1; s_off[2 * lane + 1] = incl - c1; }
    __syncthreads();
    uint32_t* keys = reinterpret_cast<uint32_t*>(sg.ws + l.samples) + s_off[way];
    for (uint32_t k = t % kWayLanes; k < mine; k += kWayLanes) keys[k] = part[k];
    __syncthreads();
    key = select_rank(reinterpret_cast<uint32_t*>(sg.ws + l.samples), found, sg.thr_index, s_hist);
  }
  // (a provisional threshold that is a NaN lets everything through: what is found at or below it is not all there is)
  if (t == 0) {
    if (key > prov) st->thr_bits = key; else st->fallback = 1;
  }
}

constexpr int kRecountWords = 32;
// What exceeds the provisional threshold but not the exact one goes: out of the lists, in place, four lanes to each; where
// the expand launch will look at the masks, because a list of its wave's is too short, out of those.
template <int CAP>
__global__ __launch_bounds__(kThreads) void gd_recount_kernel(const GdArgs<CAP> a) {
  const int blk = blockIdx.x;
  const int s = find_segment<CAP>(a.tile_start, a.nseg, blk);
  const GdSeg& sg = a.seg[s];
  const GdState* st = seg_state(sg);
  if (st->fallback) return;   // uniform
  const GdLayout l = gd_layout(sg.n, sg.sample_cnt);
  uint64_t* __restrict__ masks = reinterpret_cast<uint64_t*>(sg.ws + l.masks);
  uint32_t* __restrict__ cnt = reinterpret_cast<uint32_t*>(sg.ws + l.cnt);
  uint16_t* __restrict__ wcnt = reinterpret_cast<uint16_t*>(sg.ws + l.wcnt);
  const float* __restrict__ r = sg.r;
  const uint32_t ntiles = cdiv(sg.n, kTile);
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t group = uint32_t(blk - a.tile_start[s]), wave = threadIdx.x / kWave;
  const uint32_t tile0 = (group * (kThreads / kWave) + wave) * kListTiles;
  const uint32_t room = list_room(sg.n, sg.limit), sub = lane % kListLanes, mine = tile0 * (kThreads / kWave) + lane / kListLanes;
  const bool my_tile = tile0 + lane / (kListLanes * (kThreads / kWave)) < ntiles;
  uint2* list = seg_list(sg, l) + size_t(mine) * room;
  uint2 p[kListAhead];
  uint32_t listed = 0;
  uint32_t all = 0, big = 0;   // the wave's candidates that stay; its tiles' largest |r|
  if (lane < kListTiles && tile0 + lane < ntiles) big = reinterpret_cast<const uint32_t*>(sg.ws + l.mx)[tile0 + lane];
  if (my_tile) {
    listed = wcnt[mine];
    if (room != 0) {
#pragma unroll
      for (uint32_t q = 0; q < kListAhead; q++) p[q] = list[q * kListLanes + sub];
    }
  }
  const float thr = __uint_as_float(st->thr_bits), nthr = -thr;
  if (room != 0 && __ballot(listed > room) == 0) {
    uint32_t kept = 0;
    auto keep = [&](bool any, uint2 e) {   // kept ones move down: never past a place that is still to be read
      const float x = __uint_as_float(e.y);
      const bool k = any && (x > thr || x < nthr);
      const uint32_t group = uint32_t(__ballot(k) >> (lane - sub)) & ((1u << kListLanes) - 1u);
      if (k) list[kept + uint32_t(__popc(group & ((1u << sub) - 1u)))] = e;
      kept += uint32_t(__popc(group));
    };
#pragma unroll
    for (uint32_t q = 0; q < kListAhead; q++) keep(q * kListLanes + sub < listed, p[q]);
    for (uint32_t j = kListAhead * kListLanes; __ballot(j < listed) != 0; j += kListLanes) {
      const bool any = j + sub < listed;
      keep(any, any ? list[j + sub] : make_uint2(0, 0));
    }
    if (my_tile && sub == 0) wcnt[mine] = uint16_t(kept);
    constexpr int kTileLanes = int(kListLanes * (kThreads / kWave));
    const uint32_t c = sub == 0 ? kept : 0u;
    static_assert(kTileLanes == 16, "a tile's lists are a row of lanes");
    const uint32_t tile_cnt = row_sum(c);
    if (my_tile && lane % kTileLanes == 0) cnt[tile0 + lane / kTileLanes] = tile_cnt;
    all = wave_sum_u32(c);
  } else {
    // A mask word per lane; then its 64 elements lane by lane, kRecountWords words' values requested together: a tile full
    // of candidates takes two rounds (with each lane walking its own word's bits this launch took 29 us for the 17 M elements
    // of gd_invert_kernel's comment, now 23.5; 47.5 and 32 for its 138 M).
    uint64_t word[kListTiles];
#pragma unroll
    for (uint32_t j = 0; j < kListTiles; j++) word[j] = tile0 + j < ntiles ? masks[size_t(tile0 + j) * kWave + lane] : 0ull;
#pragma unroll 1
    for (uint32_t j = 0; j < kListTiles; j++) {
      const uint32_t tile = tile0 + j;
      const uint64_t old = j == 0 ? word[0] : j == 1 ? word[1] : j == 2 ? word[2] : word[3];
      static_assert(kListTiles == 4, "the words above");
      auto bit = [&](uint32_t w) {   // whether the lane's element of word w is a candidate
        const uint64_t m = uint64_t(uint32_t(__builtin_amdgcn_readlane(int(uint32_t(old)), int(w)))) |
                           uint64_t(uint32_t(__builtin_amdgcn_readlane(int(uint32_t(old >> 32)), int(w)))) << 32;
        return ((m >> lane) & 1ull) != 0;
      };
      uint64_t keep = 0, left = __ballot(old != 0);
      if (left == 0) continue;   // wave-uniform
      do {
        uint64_t now = left;
        float v[kRecountWords];
#pragma unroll
        for (int q = 0; q < kRecountWords; q++) {   // no branches, so that nothing is waited for in between
          const uint32_t w = left ? uint32_t(__builtin_ctzll(left)) : 0u;
          v[q] = left != 0 && bit(w) ? r[tile * uint32_t(kTile) + w * kWave + lane] : 0.0f;
          left &= left - 1;   // 0 stays 0
        }
#pragma unroll
        for (int q = 0; q < kRecountWords; q++) {
          const uint32_t w = now ? uint32_t(__builtin_ctzll(now)) : uint32_t(kWave);
          const uint64_t k = __ballot(v[q] > thr || v[q] < nthr);   // a threshold is not negative: zero does not pass
          keep = lane == w ? k : keep;
          now &= now - 1;
        }
      } while (left);
      if (keep != old) masks[size_t(tile) * kWave + lane] = keep;
      uint32_t c = uint32_t(__popcll(keep));
      c = wave_sum_u32(c);
      if (lane == 0) cnt[tile] = c;
      all += c;
    }
  }
  // The group's total and largest |r|, from which the expand launch works its places out: a scan launch before it took 6.5 us
  // of a call with its hand-over.
  __shared__ uint32_t s_all[kThreads / kWave], s_big[kThreads / kWave];
  big = wave_max_u32(big);   // zero in the other lanes
  if (lane == 0) { s_all[wave] = all; s_big[wave] = big; }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t total = 0, largest = 0;
#pragma unroll
    for (int w = 0; w < kThreads / kWave; w++) { total += s_all[w]; largest = s_big[w] > largest ? s_big[w] : largest; }
    reinterpret_cast<uint32_t*>(sg.ws + l.ctot)[group] = total;
    reinterpret_cast<uint32_t*>(sg.ws + l.cmax)[group] = largest;
  }
}

// The one pass over the tensors.  Lane l of wave w handles elements
// base + w*1024 + c*64 + l for c = 0..15, so ballot number c is the mask word of
// 64 consecutive elements in natural bit order.
// RESIDUAL = false is the sparsifier without residual (dgc_body.h:110-117): the
// values are G itself, nothing is added and nothing is stored (4 bytes per element).
// PROV: against the provisional threshold also a NaN is a candidate, as it is one of the largest of a sample.
// LISTS: some tensor of the launch may have lists.
template <bool RESIDUAL, bool PROV, bool LISTS, int CAP>
__global__ __launch_bounds__(kThreads) void gd_stream_kernel(const GdArgs<CAP> a) {
  const int tile = blockIdx.x;
  const int s = find_segment<CAP>(a.tile_start, a.nseg, tile);
  const GdSeg& sg = a.seg[s];
  const GdLayout l = gd_layout(sg.n, sg.sample_cnt);
  const float* __restrict__ g = sg.g;
  float* __restrict__ r = sg.r;
  const uint32_t n = sg.n;
  uint64_t* __restrict__ masks = reinterpret_cast<uint64_t*>(sg.ws + l.masks);
  const uint32_t t = uint32_t(tile - a.tile_start[s]);
  const float thr = __uint_as_float(seg_state(sg)->thr_bits);
  const float nthr = -thr;
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t wave = threadIdx.x / kWave;
  const uint32_t base = t * uint32_t(kTile);
  const uint32_t wbase = base + wave * uint32_t(kWaveTile);
  // The wave's candidates are also listed as they are found, values and all: the launches behind the pass would otherwise
  // fetch a line of r for each (see list_room).
  const uint32_t room = list_room(n, sg.limit);
  auto passes = [&](float x) { return PROV ? !(__builtin_fabsf(x) <= thr) : (x > thr) || (x < nthr); };  // gd_body.h:59-67
  uint2* __restrict__ list = seg_list(sg, l) + (size_t(t) * (kThreads / kWave) + wave) * room;
  uint32_t lo = 0, hi = 0, cnt = 0;
  const bool clears = LISTS && RESIDUAL && !PROV && clears_listed(n, sg.limit);
  // m: the wave's candidates of 64 elements, uniform; the result is what the element leaves in r
  auto note = [&](uint64_t m, uint32_t e, float x) {
    float left = x;
    if (LISTS && m != 0) {
      const uint32_t at = cnt + uint32_t(__popcll(m & ((1ull << lane) - 1ull)));
      if ((m >> lane & 1ull) && at < room) {
        list[at] = make_uint2(e, __float_as_uint(x));
        if (clears) left = 0.0f;
      }
    }
    cnt += uint32_t(__popcll(m));
    return left;
  };
  float big = 0.0f;  // largest |x| this lane has seen
  float gv[kPerLane], rv[kPerLane];
  if (n - base >= uint32_t(kTile)) {
#pragma unroll
    for (int c = 0; c < kPerLane; c++) {
      gv[c] = __builtin_nontemporal_load(g + size_t(wbase) + c * kWave + lane);
      rv[c] = RESIDUAL ? __builtin_nontemporal_load(r + size_t(wbase) + c * kWave + lane) : 0.0f;
    }
#pragma unroll
    for (int c = 0; c < kPerLane; c++) {
      const float x = RESIDUAL ? gv[c] + rv[c] : gv[c];  // thrust::plus<float>()(G, R), gd_body.h:121-128
      const uint64_t m = __ballot(passes(x));
      const float left = note(m, wbase + c * kWave + lane, x);
      if (RESIDUAL) __builtin_nontemporal_store(left, r + size_t(wbase) + c * kWave + lane);
      big = __builtin_fmaxf(big, __builtin_fabsf(x));
      lo = lane == uint32_t(c) ? uint32_t(m) : lo;  // lane c keeps mask word c
      hi = lane == uint32_t(c) ? uint32_t(m >> 32) : hi;
    }
  } else {
    // The tile that holds the end of the tensor: all its loads first, as above (a load, add, store per
    // step would make this one workgroup wait for memory sixteen times in a row at the very end of the launch).
#pragma unroll
    for (int c = 0; c < kPerLane; c++) {
      const uint32_t e = wbase + c * kWave + lane;
      gv[c] = e < n ? g[e] : 0.0f;
      rv[c] = (RESIDUAL && e < n) ? r[e] : 0.0f;
    }
#pragma unroll
    for (int c = 0; c < kPerLane; c++) {
      const uint32_t e = wbase + c * kWave + lane;
      bool p = false;
      const float x = RESIDUAL ? gv[c] + rv[c] : gv[c];
      if (e < n) {
        p = passes(x);
        big = __builtin_fmaxf(big, __builtin_fabsf(x));
      }
      const uint64_t m = __ballot(p);
      const float left = note(m, e, x);
      if (RESIDUAL && e < n) r[e] = left;
      lo = lane == uint32_t(c) ? uint32_t(m) : lo;  // lane c keeps mask word c
      hi = lane == uint32_t(c) ? uint32_t(m >> 32) : hi;
    }
  }
  if (lane < kPerLane) masks[(size_t(wbase) >> 6) + lane] = (uint64_t(hi) << 32) | lo;
  if (PROV && cnt > room && lane == 0) seg_state(sg)->crowded = 1;   // all of them store the same
  // which of the wave's sixteen mask words have a bit set (lanes beyond the sixteenth hold zeros)
  const uint32_t any16 = uint32_t(__ballot((lo | hi) != 0u));
  uint32_t bigb = __float_as_uint(big);  // non-negative floats order like their bit patterns; a NaN is not an input
  bigb = wave_max_u32(bigb);
  __shared__ uint32_t s_cnt[kThreads / kWave], s_big[kThreads / kWave], s_any[kThreads / kWave];
  if (lane == 0) { s_cnt[wave] = cnt; s_big[wave] = bigb; s_any[wave] = any16; }
  __syncthreads();
  if (threadIdx.x == 0) {
    reinterpret_cast<uint32_t*>(sg.ws + l.cnt)[t] = s_cnt[0] + s_cnt[1] + s_cnt[2] + s_cnt[3];
    if (LISTS) reinterpret_cast<uint64_t*>(sg.ws + l.wcnt)[t] =
        uint64_t(s_cnt[0]) | (uint64_t(s_cnt[1]) << 16) | (uint64_t(s_cnt[2]) << 32) | (uint64_t(s_cnt[3]) << 48);
    reinterpret_cast<uint64_t*>(sg.ws + l.coarse)[t] =
        uint64_t(s_any[0]) | (uint64_t(s_any[1]) << 16) | (uint64_t(s_any[2]) << 32) | (uint64_t(s_any[3]) << 48);
    const uint32_t m01 = s_big[0] > s_big[1] ? s_big[0] : s_big[1], m23 = s_big[2] > s_big[3] ? s_big[2] : s_big[3];
    reinterpret_cast<uint32_t*>(sg.ws + l.mx)[t] = m01 > m23 ? m01 : m23;
  }
}

// Exclusive prefix of the per-tile counts within chunks of 4096 tiles: workgroup c of a tensor scans counts
// [c*4096, (c+1)*4096) into `off` (relative to its chunk) and leaves the chunk's total and largest |r|.
// The second level - at most 128 chunk totals per tensor - is folded by the expand launch itself, each
// wave for its own tiles, so no workgroup here waits for or counts the others.
template <int CAP>
__global__ __launch_bounds__(kSelThreads) void gd_scan_kernel(const GdArgs<CAP> a) {
  __shared__ uint32_t s_wave[kSelThreads / kWave], s_wmax[kSelThreads / kWave];
  const int tile = blockIdx.x;
  const int s = find_segment<CAP>(a.tile_start, a.nseg, tile);
  const GdSeg& sg = a.seg[s];
  const GdLayout l = gd_layout(sg.n, sg.sample_cnt);
  const uint32_t* __restrict__ cnt = reinterpret_cast<const uint32_t*>(sg.ws + l.cnt);
  const uint32_t* __restrict__ mxs = reinterpret_cast<const uint32_t*>(sg.ws + l.mx);
  uint32_t* __restrict__ off = reinterpret_cast<uint32_t*>(sg.ws + l.off);
  uint32_t* chunk_tot = reinterpret_cast<uint32_t*>(sg.ws + l.ctot);
  uint32_t* chunk_max = reinterpret_cast<uint32_t*>(sg.ws + l.cmax);
  const uint32_t n = cdiv(sg.n, kTile);                                   // tiles of this tensor
  const uint32_t chunk = uint32_t(tile - a.tile_start[s]);
  const uint32_t t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
  const uint32_t i0 = chunk * uint32_t(kScanChunk) + t * 4;
  uint32_t c[4], big = 0;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    c[j] = (i0 + j < n) ? cnt[i0 + j] : 0u;
    const uint32_t m = (i0 + j < n) ? mxs[i0 + j] : 0u;
    big = m > big ? m : big;
  }
  const uint32_t sum = c[0] + c[1] + c[2] + c[3];
  const uint32_t incl = wave_prefix_u32(sum);
  big = wave_max_u32(big);
  if (lane == kWave - 1) { s_wave[wave] = incl; s_wmax[wave] = big; }
  __syncthreads();
  uint32_t before = 0, all = 0, allmax = 0;
#pragma unroll
  for (uint32_t w = 0; w < kSelThreads / kWave; w++) {
    const uint32_t v = s_wave[w];
    if (w < wave) before += v;
    all += v;
    allmax = s_wmax[w] > allmax ? s_wmax[w] : allmax;
  }
  uint32_t run = before + incl - sum;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    if (i0 + j < n) off[i0 + j] = run;
    run += c[j];
  }
  if (t == 0) {
    chunk_tot[chunk] = all;
    chunk_max[chunk] = allmax;
  }
}

// Tensors of at most kScanChunk tiles (16.7 M elements), and those of the provisional path, whose recount leaves totals of 16
// tiles each, take no part in the scan launch: the expand launch's
// workgroups add up the counts before their tiles for themselves (at most 16 KB out of the L2), which saves
// a launch of 3-5 us.
//
// Turns the per-tile bit masks into the ascending index list, kExpandTiles consecutive tiles
// per wave (their mask words, and then the values of their first candidates, are loaded
// together: a wave with one tile spent its time waiting for one load after the other, and
// the launch needed four rounds of such waves), at the offsets the scan produced.  Every wave
// folds the chunk totals for itself (at most 128 of them): the offset of its tiles' chunks and the
// tensor's candidate count; the wave of a tensor's first tile reports count, threshold and
// largest |r| to the host.  If the stream pass found at most `limit`
// candidates this is the finish (gd_body.h:193-229): indices, values and header
// are written and the residual entries cleared.  If it found more, the candidates
// and their keys (bits of |r|) go to the cut path's buffers instead and
// nothing else is touched; more than `cap` candidates do not fit those buffers
// and the kernel does nothing for that tensor (the host then calls it again with larger ones,
// limit = 0 and no report).
constexpr int kExpandTiles = int(kListTiles);
constexpr int kExpandPerBlock = (kThreads / kWave) * kExpandTiles;  // tiles per workgroup
static_assert(kExpandPerBlock == kGroupTiles && kExpandTiles == int(kListTiles), "the recount's groups are these workgroups' tiles");
template <int CAP>
__global__ __launch_bounds__(kThreads) void gd_expand_kernel(const GdArgs<CAP> a) {
  const int blk = blockIdx.x;
  const int s = find_segment<CAP>(a.tile_start, a.nseg, blk);
  const GdSeg& sg = a.seg[s];
  const GdLayout l = gd_layout(sg.n, sg.sample_cnt);
  const CutLayout cl = cut_layout(sg.cap);
  const GdState* st = seg_state(sg);
  const uint64_t* __restrict__ masks = reinterpret_cast<const uint64_t*>(sg.ws + l.masks);
  const uint32_t* __restrict__ tile_off = reinterpret_cast<const uint32_t*>(sg.ws + l.off);
  const uint32_t* __restrict__ chunk_tot = reinterpret_cast<const uint32_t*>(sg.ws + l.ctot);
  uint8_t* __restrict__ out = sg.out;
  float* __restrict__ r = sg.r;
  const uint32_t ntiles = cdiv(sg.n, kTile);
  const uint32_t nchunks = cdiv(ntiles, kScanChunk);
  const uint32_t lane = threadIdx.x & (kWave - 1);
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t tile0 = (uint32_t(blk - a.tile_start[s]) * (kThreads / kWave) + wave) * kExpandTiles;

  // The lists of this wave's tiles.
  constexpr uint32_t kPer = kListLanes, kAhead = kListAhead;
  const uint32_t room = list_room(sg.n, sg.limit ? sg.limit : a.listed);
  const uint32_t sub = lane % kPer, mine_list = tile0 * (kThreads / kWave) + lane / kPer;
  const bool my_tile = tile0 + lane / (kPer * (kThreads / kWave)) < ntiles;
  const uint2* __restrict__ list = seg_list(sg, l) + size_t(mine_list) * room;
  uint2 first[kAhead];
  uint32_t listed = 0;
  if (room != 0 && my_tile) {
    listed = reinterpret_cast<const uint16_t*>(sg.ws + l.wcnt)[mine_list];
#pragma unroll
    for (uint32_t q = 0; q < kAhead; q++) first[q] = list[q * kPer + sub];
  }

  __shared__ uint32_t s_sum[3][kThreads / kWave];
  uint32_t total, mm = 0;      // the tensor's candidates; its largest |r| (only the wave that reports needs it)
  uint32_t ex0 = 0, ex1 = 0;   // scanned tensors: exclusive prefixes of chunks 2 * lane and 2 * lane + 1
  uint32_t own_off = 0;        // the others: lane j's tile tile0 + j starts here
  const bool grouped = a.margin >= 0;   // the recount has left the totals of the workgroups' tiles
  const bool scanned = nchunks > 1 && !grouped;
  if (scanned) {
    // chunk totals, two per lane: inclusive prefix over the lanes
    const uint32_t* __restrict__ chunk_max = reinterpret_cast<const uint32_t*>(sg.ws + l.cmax);
    const uint32_t a0 = 2 * lane < nchunks ? chunk_tot[2 * lane] : 0u, a1 = 2 * lane + 1 < nchunks ? chunk_tot[2 * lane + 1] : 0u;
    const uint32_t inc2 = wave_prefix_u32(a0 + a1);
    total = __builtin_amdgcn_readlane(inc2, kWave - 1);
    ex0 = inc2 - a0 - a1;
    ex1 = ex0 + a0;
    if (tile0 == 0) {
      const uint32_t m0 = 2 * lane < nchunks ? chunk_max[2 * lane] : 0u, m1 = 2 * lane + 1 < nchunks ? chunk_max[2 * lane + 1] : 0u;
      mm = m0 > m1 ? m0 : m1;
      mm = wave_max_u32(mm);
    }
  } else {
    // The counts of all tiles, or of all groups, four per lane and load (the array's padding may be read, not used): the
    // total, and what lies before this workgroup's first tile.
    const uint32_t own_group = uint32_t(blk - a.tile_start[s]);
    const uint32_t first = grouped ? own_group : own_group * kExpandPerBlock, counts = grouped ? cdiv(ntiles, kGroupTiles) : ntiles;
    const uint4* __restrict__ cnt4 = reinterpret_cast<const uint4*>(sg.ws + (grouped ? l.ctot : l.cnt));
    const uint4* __restrict__ mx4 = reinterpret_cast<const uint4*>(sg.ws + (grouped ? l.cmax : l.mx));
    constexpr uint32_t kSteps = kScanChunk / (4 * kThreads);
    const uint32_t j = tile0 + lane;
    const uint32_t mine = lane < uint32_t(kExpandTiles) && j < ntiles ? reinterpret_cast<const uint32_t*>(sg.ws + l.cnt)[j] : 0u;
    uint32_t all = 0, before = 0;
#pragma unroll 1
    for (uint32_t i0 = 0; i0 < counts; i0 += kScanChunk) {   // once, up to 2^24 elements, on the provisional path 2^28
      uint4 c[kSteps], big[kSteps];
#pragma unroll
      for (uint32_t q = 0; q < kSteps; q++) {
        const uint32_t i = i0 / 4 + q * kThreads + threadIdx.x;
        const bool any = 4 * i < counts;
        c[q] = any ? cnt4[i] : make_uint4(0, 0, 0, 0);
        big[q] = any && first == 0 ? mx4[i] : make_uint4(0, 0, 0, 0);
      }
#pragma unroll
      for (uint32_t q = 0; q < kSteps; q++) {
        const uint32_t i = i0 + 4 * (q * kThreads + threadIdx.x);
        const uint32_t v[4] = {c[q].x, c[q].y, c[q].z, c[q].w}, b[4] = {big[q].x, big[q].y, big[q].z, big[q].w};
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) {
          const uint32_t x = i + k < counts ? v[k] : 0u, y = i + k < counts ? b[k] : 0u;
          all += x;
          before += i + k < first ? x : 0u;
          mm = y > mm ? y : mm;
        }
      }
    }
    all = wave_sum_u32(all);
    before = wave_sum_u32(before);
    mm = wave_max_u32(mm);
    const uint32_t incl = wave_prefix_u32(mine);
    const uint32_t own = __builtin_amdgcn_readlane(incl, kExpandTiles - 1);  // this wave's candidates
    __shared__ uint32_t s_own[kThreads / kWave];
    if (lane == 0) { s_sum[0][wave] = all; s_sum[1][wave] = before; s_sum[2][wave] = mm; s_own[wave] = own; }
    __syncthreads();
    total = 0;
    own_off = incl - mine;
    mm = 0;
#pragma unroll
    for (uint32_t w = 0; w < kThreads / kWave; w++) {
      total += s_sum[0][w];
      own_off += s_sum[1][w] + (w < wave ? s_own[w] : 0u);
      mm = s_sum[2][w] > mm ? s_sum[2][w] : mm;
    }
  }
  if (a.margin >= 0 && st->fallback) {
    // the provisional threshold lies above the exact one: nothing of what the masks hold may be used
    if (tile0 == 0 && a.report != nullptr && lane == 0) {
      uint32_t* rep = a.report + size_t(s) * kReportWords;
      __hip_atomic_store(rep + 0, kFallback, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      __hip_atomic_store(rep + 1, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      __hip_atomic_store(rep + 2, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    return;
  }
  const bool cut_here = a.device_cut != 0 && sg.limit < kCutKeep;
  if (tile0 == 0 && lane == 0) seg_state(sg)->total = total;
  if (tile0 == 0 && a.report != nullptr && !cut_here) {
    // Pinned host words the host polls (no copy command, no wait for the stream).  The host waits for each
    // of the three words to change, so plain system-scope stores do (a release would write the whole L2 back).
    if (lane == 0) {
      uint32_t* rep = a.report + size_t(s) * kReportWords;
      __hip_atomic_store(rep + 0, total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      __hip_atomic_store(rep + 1, st->thr_bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      __hip_atomic_store(rep + 2, mm, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
  const bool cut = total > sg.limit;
  if (cut && total > sg.cap) return;
  if (!cut && tile0 == 0 && lane == 0) *reinterpret_cast<int32_t*>(out) = int32_t(4 + total * 8);
  if (tile0 >= ntiles) return;

  const uint32_t thr_bits = st->thr_bits;
  int32_t* __restrict__ cand = reinterpret_cast<int32_t*>(sg.cut + cl.ia);
  uint32_t* __restrict__ keys = reinterpret_cast<uint32_t*>(sg.cut + cl.ka);
  // In a cut the sign travels in the index's top bit: no launch then has to read the values again.
  const uint32_t sign = 0x80000000u;
  int32_t* idx = reinterpret_cast<int32_t*>(out + 4);
  float* val = reinterpret_cast<float*>(out + 4 + size_t(total) * 4);
  if (room != 0 && __ballot(listed > room) == 0) {
    // All of the wave's candidates are in its lists: the tiles follow each other, so one prefix over the lists' lengths is
    // every list's place.
    const uint32_t own = sub == 0 ? listed : 0u;
    const uint32_t incl = wave_prefix_u32(own);
    const uint32_t chunk = tile0 / kScanChunk;
    static_assert(kScanChunk % kExpandTiles == 0, "a wave's tiles are of one chunk");
    const uint32_t start = scanned ? uint32_t(__builtin_amdgcn_readlane(int((chunk & 1u) ? ex1 : ex0), int(chunk >> 1))) + tile_off[tile0]
                                   : uint32_t(__builtin_amdgcn_readlane(own_off, 0));
    static_assert(kPer == 4, "a list's lanes are a quad");
    const uint32_t at = start + uint32_t(__builtin_amdgcn_update_dpp(0, int(incl - own), 0x00, 0xF, 0xF, false));   // of the quad's first lane
    auto put = [&](uint32_t place, uint2 p) {
      if (cut) {
        cand[place] = int32_t(p.x | (p.y & sign));
        keys[place] = (p.y & 0x7FFFFFFFu) - thr_bits;
      } else {
        idx[place] = int32_t(p.x);
        val[place] = __uint_as_float(p.y);
        r[p.x] = 0.0f;
      }
    };
#pragma unroll
    for (uint32_t q = 0; q < kAhead; q++)
      if (q * kPer + sub < listed) put(at + q * kPer + sub, first[q]);
    for (uint32_t j = kAhead * kPer + sub; j < listed; j += kPer) put(at + j, list[j]);
    return;
  }
  // Through the masks.
  uint64_t m[kExpandTiles];
#pragma unroll
  for (int j = 0; j < kExpandTiles; j++) m[j] = tile0 + j < ntiles ? masks[size_t(tile0 + j) * kWave + lane] : 0ull;
  // first place of every tile's candidates, then of this lane's within the tile
  uint32_t pos[kExpandTiles];
#pragma unroll
  for (int j = 0; j < kExpandTiles; j++) {
    const uint32_t tile = tile0 + j < ntiles ? tile0 + j : ntiles - 1;
    const uint32_t chunk = tile / kScanChunk;
    const uint32_t start = scanned ? uint32_t(__builtin_amdgcn_readlane(int((chunk & 1u) ? ex1 : ex0), int(chunk >> 1))) + tile_off[tile]
                                   : uint32_t(__builtin_amdgcn_readlane(own_off, j));
    const uint32_t c = __popcll(m[j]);
    const uint32_t incl = wave_prefix_u32(c);
    pos[j] = start + incl - c;
  }
  // The first candidate of each of the lane's 64-element groups: their values are loaded together.
  uint32_t e1[kExpandTiles];
  float v1[kExpandTiles];
#pragma unroll
  for (int j = 0; j < kExpandTiles; j++) {
    e1[j] = (tile0 + j) * uint32_t(kTile) + lane * kWave + uint32_t(m[j] ? __builtin_ctzll(m[j]) : 0);
    v1[j] = m[j] ? r[e1[j]] : 0.0f;
  }
  if (cut) {
    // Sort key: distance of |r| above the threshold in fp32 bit patterns (same order as |r|;
    // the high digits of such keys are mostly zero, which lets the sort skip its last passes).
#pragma unroll
    for (int j = 0; j < kExpandTiles; j++) {
      if (m[j]) {
        cand[pos[j]] = int32_t(e1[j] | (__float_as_uint(v1[j]) & sign));
        keys[pos[j]] = __float_as_uint(__builtin_fabsf(v1[j])) - thr_bits;
        pos[j]++;
        m[j] &= m[j] - 1;
      }
      const uint32_t e0 = (tile0 + j) * uint32_t(kTile) + lane * kWave;
      while (m[j]) {  // further candidates of the same group: rare
        const uint32_t e = e0 + uint32_t(__builtin_ctzll(m[j]));
        m[j] &= m[j] - 1;
        const float v = r[e];
        cand[pos[j]] = int32_t(e | (__float_as_uint(v) & sign));
        keys[pos[j]] = __float_as_uint(__builtin_fabsf(v)) - thr_bits;
        pos[j]++;
      }
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < kExpandTiles; j++) {
    if (m[j]) {
      idx[pos[j]] = int32_t(e1[j]);
      val[pos[j]] = v1[j];
      r[e1[j]] = 0.0f;
      pos[j]++;
      m[j] &= m[j] - 1;
    }
    const uint32_t e0 = (tile0 + j) * uint32_t(kTile) + lane * kWave;
    while (m[j]) {
      const uint32_t e = e0 + uint32_t(__builtin_ctzll(m[j]));
      m[j] &= m[j] - 1;
      idx[pos[j]] = int32_t(e);
      val[pos[j]] = r[e];
      r[e] = 0.0f;
      pos[j]++;
    }
  }
}

// ---- cut to the `expected` largest |r| (gd_body.h:176-187) ------------------
// Stable LSD radix sort of (key, index) pairs, 8 or 9 bits per pass (9 when that
// saves a pass: keys of 25 to 27 bits, as the configuration's heavy-tailed gradient
// gives, take three passes instead of four), descending (bin = BINS - 1 - digit).
// A pass is a count launch and a scatter launch over tiles of 4096 pairs
// (1024 lanes x 4), counts[tile * BINS + bin]; the last pass writes
// the message instead of a sorted list.  All tensors of a call that
// have to be cut share these launches (a table of tensors in the kernel arguments);
// the number of passes is that of the tensor with the largest key (a pass over a
// digit that is zero in every key of a tensor leaves that tensor's order as it is).
// (All passes in one launch
// with grid-wide barriers was tried and lost: data handed between workgroups
// inside a launch needs device-scope accesses or whole-L2 fences, either of
// which costs more than the launches saved.)  (Counting a pass's digits where its
// input is written, with global atomics, saves the count launches but was five
// times slower: some 10^5 scattered atomics cost more than the launches.)
struct SortSeg {           // one tensor that is being cut; 40 bytes
  uint8_t* cut;            // its buffers, cut_layout(cap): the pass with parity p reads one copy of keys and indices and writes the other
  uint8_t* msg;            // the message, which the last pass writes
  float* r;                // the entries that are sent are cleared here
  uint32_t n;              // candidates
  uint32_t keep;           // `expected`
  uint32_t cap;
  uint32_t thr_bits;       // a candidate's key is |r| less this, as bits
};
static_assert(sizeof(SortSeg) == 40, "segment record");
__device__ __forceinline__ uint32_t* sort_keys(const SortSeg& sg, const CutLayout& c, int parity) {
  return reinterpret_cast<uint32_t*>(sg.cut + (parity ? c.kb : c.ka));
}
__device__ __forceinline__ int32_t* sort_ids(const SortSeg& sg, const CutLayout& c, int parity) {
  return reinterpret_cast<int32_t*>(sg.cut + (parity ? c.ib : c.ia));
}
__device__ __forceinline__ uint32_t* sort_counts(const SortSeg& sg, const CutLayout& c) {   // [tile][bins] of the current pass
  return reinterpret_cast<uint32_t*>(sg.cut + c.sc);
}
template <int CAP>
struct SortArgs {
  int32_t nseg;
  int32_t shift;
  int32_t parity;
  int32_t last;            // this pass writes the messages
  int32_t tile_start[CAP + 1];
  SortSeg seg[CAP];
};
static_assert(sizeof(SortArgs<kCapLarge>) <= 18000, "kernel-argument budget");

// Lanes of the wave whose `bin` equals this lane's, among the lanes in `live`.
template <int BITS>
__device__ __forceinline__ uint64_t match_bin(uint32_t bin, bool live) {
  uint64_t same = __ballot(live);
#pragma unroll
  for (int b = 0; b < BITS; b++) {
    const uint64_t m = __ballot((bin >> b) & 1u);
    same &= ((bin >> b) & 1u) ? m : ~m;
  }
  return same;
}

// One LDS atomic per distinct bin of a wave's 64 keys, not one per key: the top
// digit of keys that are all just above one threshold is the same for nearly all
// of them, and 8192 atomics on one LDS word took longer than the rest of the pass.
template <int CAP, int BITS>
__global__ __launch_bounds__(kSortThreads) void gd_sort_count_kernel(const SortArgs<CAP> a) {
  constexpr uint32_t BINS = 1u << BITS;
  const int tile = blockIdx.x;
  const int s = find_segment<CAP>(a.tile_start, a.nseg, tile);
  const SortSeg& sg = a.seg[s];
  const CutLayout cl = cut_layout(sg.cap);
  const uint32_t* __restrict__ keys = sort_keys(sg, cl, a.parity);
  const uint32_t n = sg.n;
  const int shift = a.shift;
  const uint32_t ltile = uint32_t(tile - a.tile_start[s]);
  uint32_t* __restrict__ counts = sort_counts(sg, cl);
  __shared__ uint32_t s_hist[BINS];
  const uint32_t t = threadIdx.x;
  const uint32_t lane = t & (kWave - 1);
  if (t < BINS) s_hist[t] = 0;
  const uint32_t b0 = ltile * uint32_t(kSortTile);
  uint32_t key[kSortPer];
#pragma unroll
  for (int j = 0; j < kSortPer; j++) {
    const uint32_t x = b0 + j * kSortThreads + t;
    key[j] = x < n ? keys[x] : 0u;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kSortPer; j++) {
    const bool live = b0 + j * kSortThreads + t < n;
    const uint32_t bin = (BINS - 1) - ((key[j] >> shift) & (BINS - 1));
    const uint64_t same = match_bin<BITS>(bin, live);
    if (live && (same & ((uint64_t(1) << lane) - 1)) == 0) atomicAdd(&s_hist[bin], uint32_t(__popcll(same)));
  }
  __syncthreads();
  if (t < BINS) counts[size_t(ltile) * BINS + t] = s_hist[t];
}

// A wave owns 256 consecutive pairs of the tile and takes them 64 at a time, so
// the order wave, round, lane is the input order and equal digits keep it.  Per
// round the lanes of a wave that share a bin are found with ballots; the wave
// keeps its own running count per bin in its row of s_cnt (no workgroup barrier
// inside the loop).  One pass over the 16 rows gives every wave its first place
// per bin within the tile; the pairs are then put in that order in LDS, so that
// consecutive lanes write consecutive slots of a bin's run (scattering straight
// from registers costs one address per lane and made the pass twice as long).
template <int CAP, int BITS>
__global__ __launch_bounds__(kSortThreads) void gd_sort_pass_kernel(const SortArgs<CAP> a) {
  constexpr uint32_t BINS = 1u << BITS;
  constexpr uint32_t kBinWaves = BINS / kWave;    // waves whose lanes each look after one bin
  extern __shared__ __align__(16) uint32_t s_stage[];          // [kSortTile] keys, then [kSortTile] indices
  __shared__ uint32_t s_cnt[kSortWaves][BINS];   // per wave: pairs per bin, then the wave's first place per bin
  __shared__ uint32_t s_first[BINS];             // first place of the bin within the tile
  __shared__ uint32_t s_slot[BINS];              // first global slot of the bin's pairs of this tile
  __shared__ uint32_t s_part[2 * kBinWaves];
  uint32_t* s_key = s_stage;
  uint32_t* s_id = s_stage + kSortTile;
  const uint32_t t = threadIdx.x;
  const uint32_t lane = t & (kWave - 1), wave = t / kWave;
  const int gtile = blockIdx.x;
  const int sgi = find_segment<CAP>(a.tile_start, a.nseg, gtile);
  const SortSeg& sg = a.seg[sgi];
  const uint32_t n = sg.n;
  const uint32_t blk = uint32_t(gtile - a.tile_start[sgi]);                         // this tensor's tile ...
  const uint32_t nblk = uint32_t(a.tile_start[sgi + 1] - a.tile_start[sgi]);       // ... of so many
  const CutLayout cl = cut_layout(sg.cap);
  const uint32_t* __restrict__ keys_in = sort_keys(sg, cl, a.parity);
  const int32_t* __restrict__ idx_in = sort_ids(sg, cl, a.parity);
  uint32_t* __restrict__ keys_out = sort_keys(sg, cl, 1 - a.parity);
  int32_t* __restrict__ idx_out = sort_ids(sg, cl, 1 - a.parity);
  const uint32_t* __restrict__ counts = sort_counts(sg, cl);
  // The last pass writes the message (generate_S_value, gd_body.h:80-99, and the header, :193-201): a pair is all of an
  // entry, its value the key above the threshold and the sign in the index's top bit, so nothing of r is read, and its
  // clearing is a store that nobody waits for.  (A launch behind it that looked the values up: 9 us for 138 thousand
  // entries of 138 M elements, 42 for 760 thousand of 76 M; the last pass takes 6 and 24 longer.)
  uint8_t* __restrict__ msg = a.last ? sg.msg : nullptr;
  const uint32_t keep = sg.keep, thr_bits = sg.thr_bits;
  float* __restrict__ r = sg.r;
  auto send = [&](uint32_t slot, uint32_t k, uint32_t i) {
    const uint32_t at = i & 0x7FFFFFFFu;
    reinterpret_cast<uint32_t*>(msg + 4)[slot] = at;
    reinterpret_cast<uint32_t*>(msg + 4 + size_t(keep) * 4)[slot] = (k + thr_bits) | (i & 0x80000000u);
    r[at] = 0.0f;
  };
  if (msg && blk == 0 && t == 0) *reinterpret_cast<int32_t*>(msg) = int32_t(4 + keep * 8);
  const uint32_t b0 = blk * uint32_t(kSortTile);
  const uint32_t x0 = b0 + wave * uint32_t(kSortPer * kWave) + lane;
  uint32_t key[kSortPer];
  int32_t id[kSortPer];
#pragma unroll
  for (int j = 0; j < kSortPer; j++) {
    const uint32_t x = x0 + j * kWave;
    key[j] = x < n ? keys_in[x] : 0u;
    id[j] = x < n ? idx_in[x] : 0;
  }
  // bin t (first BINS lanes): pairs in all tiles, in the tiles before this one, in this one.
  // Up to 40 tiles (163,840 pairs) are read with independent loads.
  uint32_t total = 0, before = 0, mine = 0;
  constexpr uint32_t kFlat = 40;
  if (nblk <= kFlat) {
    if (t < BINS) {
      uint32_t c[kFlat];
#pragma unroll
      for (uint32_t q = 0; q < kFlat; q++) c[q] = q < nblk ? counts[size_t(q) * BINS + t] : 0u;
#pragma unroll
      for (uint32_t q = 0; q < kFlat; q++) {
        total += c[q];
        before += q < blk ? c[q] : 0u;
        mine += q == blk ? c[q] : 0u;
      }
    }
  } else {
    // More tiles: shared out over all lanes, sixteen loads in flight in each (one bin's lane on its own, load after load,
    // made a pass over 760 K pairs 43 us long; now 13).
    constexpr uint32_t kShare = uint32_t(kSortThreads) / BINS, kRound = 16;
    const uint32_t b = t % BINS, g = t / BINS;
    for (uint32_t q0 = g; q0 < nblk; q0 += kShare * kRound) {
      uint32_t c[kRound];
#pragma unroll
      for (uint32_t k = 0; k < kRound; k++) c[k] = q0 + k * kShare < nblk ? counts[size_t(q0 + k * kShare) * BINS + b] : 0u;
#pragma unroll
      for (uint32_t k = 0; k < kRound; k++) {
        total += c[k];
        before += q0 + k * kShare < blk ? c[k] : 0u;
        mine += q0 + k * kShare == blk ? c[k] : 0u;
      }
    }
    s_stage[t] = total;
    s_stage[kSortThreads + t] = before;
    s_stage[2 * kSortThreads + t] = mine;
    __syncthreads();
    total = before = mine = 0;
    if (t < BINS) {
#pragma unroll
      for (uint32_t k = 0; k < kShare; k++) {
        total += s_stage[k * BINS + t];
        before += s_stage[kSortThreads + k * BINS + t];
        mine += s_stage[2 * kSortThreads + k * BINS + t];
      }
    }
    __syncthreads();
  }
  if (msg) {
    // Last pass: if every key has the same digit the input is already in order.
    if (__syncthreads_or(t < BINS && total == n)) {
#pragma unroll
      for (int j = 0; j < kSortPer; j++) {
        const uint32_t x = x0 + j * kWave;
        if (x < n && x < keep) send(x, key[j], uint32_t(id[j]));
      }
      return;
    }
  }
#pragma unroll
  for (uint32_t q = 0; q < kBinWaves; q++) s_cnt[wave][q * kWave + lane] = 0;  // own row: no barrier needed before use

  uint32_t place[kSortPer], bin[kSortPer];
#pragma unroll
  for (int j = 0; j < kSortPer; j++) {
    const bool live = x0 + j * kWave < n;
    bin[j] = (BINS - 1) - ((key[j] >> a.shift) & (BINS - 1));
    const uint64_t same = match_bin<BITS>(bin[j], live);
    const uint32_t rank = __popcll(same & ((uint64_t(1) << lane) - 1));
    uint32_t base = 0;
    if (live && rank == 0) {
      base = s_cnt[wave][bin[j]];
      s_cnt[wave][bin[j]] = base + uint32_t(__popcll(same));
    }
    base = __shfl(base, live ? __builtin_ctzll(same) : int(lane), kWave);
    place[j] = base + rank;
  }

  // Exclusive scans over the bins, of the global totals and of this tile's
  // counts: within each of the first BINS / 64 waves, then across them.
  const uint32_t incl_g = wave_prefix_u32(total), incl_l = wave_prefix_u32(mine);
  if (t < BINS && lane == kWave - 1) { s_part[wave] = incl_g; s_part[kBinWaves + wave] = incl_l; }
  __syncthreads();  // also: every wave's row of s_cnt is complete
  if (t < BINS) {
    uint32_t slot = incl_g - total + before, first = incl_l - mine;
    for (uint32_t w = 0; w < wave; w++) { slot += s_part[w]; first += s_part[kBinWaves + w]; }
    s_slot[t] = slot;
    s_first[t] = first;
    uint32_t run = first;
#pragma unroll
    for (int w = 0; w < kSortWaves; w++) {
      const uint32_t c = s_cnt[w][t];
      s_cnt[w][t] = run;
      run += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kSortPer; j++) {
    if (x0 + j * kWave < n) {
      const uint32_t p = s_cnt[wave][bin[j]] + place[j];
      s_key[p] = key[j];
      s_id[p] = uint32_t(id[j]);
    }
  }
  __syncthreads();
  const uint32_t live_n = n - b0 < uint32_t(kSortTile) ? n - b0 : uint32_t(kSortTile);
#pragma unroll
  for (int j = 0; j < kSortPer; j++) {
    const uint32_t p = j * kSortThreads + t;
    if (p < live_n) {
      const uint32_t k = s_key[p];
      const int32_t i = int32_t(s_id[p]);
      const uint32_t b = (BINS - 1) - ((k >> a.shift) & (BINS - 1));
      const uint32_t slot = s_slot[b] + (p - s_first[b]);
      if (msg) {
        if (slot < keep) send(slot, k, uint32_t(i));
      } else {
        keys_out[slot] = k;
        idx_out[slot] = i;
      }
    }
  }
}

// The sixteen waves' sums, folded: what lies before this wave's, and all of them.  A row of lanes reads them and shifts them
// through itself.  (Sixteen waves on one CU: an instruction of each takes a SIMD sixteen cycles, so a hundred and fifty take a
// microsecond.  Every wave walking the sixteen words took sixty.)
__device__ __forceinline__ uint32_t before_wave(uint32_t sum_of_lane, uint32_t& total) {
  static_assert(kSortWaves == 16, "a row of lanes");
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x / kWave));
  const uint32_t incl = row_prefix_u32(sum_of_lane);
  total = uint32_t(__builtin_amdgcn_readlane(int(incl), 15));
  return uint32_t(__builtin_amdgcn_readlane(int(incl - sum_of_lane), wave));
}
// Exclusive prefix of `v` over the workgroup's lanes in order; `total` is the sum.  s_wave: a word per wave.
__device__ __forceinline__ uint32_t block_prefix(uint32_t v, uint32_t* s_wave, uint32_t& total) {
  const uint32_t lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const uint32_t incl = wave_prefix_u32(v);
  if (lane == kWave - 1) s_wave[wave] = incl;
  __syncthreads();
  const uint32_t before = before_wave(s_wave[lane & 15], total);
  __syncthreads();
  return before + incl - v;
}
// The same with one barrier, for words of `s_wave` that nobody uses again before the next one; `any`: whether some lane's flag
// is set (a wave's sum is below 2^31).
__device__ __forceinline__ uint32_t block_prefix_once(uint32_t v, bool flag, uint32_t* s_wave, uint32_t& total, bool& any) {
  const uint32_t lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const uint32_t incl = wave_prefix_u32(v);
  const uint32_t marked = __ballot(flag) != 0 ? 0x80000000u : 0u;
  if (lane == kWave - 1) s_wave[wave] = incl | marked;
  __syncthreads();
  const uint32_t c = s_wave[lane & 15];
  any = __ballot((c >> 31) != 0) != 0;
  return before_wave(c & 0x7FFFFFFFu, total) + incl - v;
}

// The `keep` largest |r| among the elements whose mask bit is set, in ascending index order, to LDS (keys as
// distances from the threshold, the sign in the index's top bit): for a tensor with more candidates than fit.  A rank search over the candidates, then
// one walk that lists those above the value found and the first ones equal to it.  Slow (one workgroup, four
// walks over the mask) and all but never needed: a sampled threshold lets twice the expected number
// through only where the sample is a handful of values.  (While the workgroup held 8192 pairs, every other cut of a
// tensor that keeps nearly as many came here: 23 tensors of 16.5 M, one in a hundred kept, 122-137 us; now 50-64.)
__device__ __forceinline__ void top_of_masks(const uint64_t* __restrict__ masks, const float* __restrict__ r, uint32_t n, uint32_t keep,
                                             uint32_t thr_bits, uint32_t* s_hist, uint32_t* s_wave, uint32_t* s_key, uint32_t* s_id) {
  const uint32_t words = cdiv(n, kWave), t = threadIdx.x;
  uint32_t prefix = 0, rank = keep - 1;
#pragma unroll 1
  for (int pass = 1; pass <= 3; pass++) {
    for (int i = t; i < kBins1; i += kSortThreads) s_hist[i] = 0;
    __syncthreads();
    for (uint32_t w = t; w < words; w += kSortThreads) {
      for (uint64_t m = masks[w]; m; m &= m - 1) {
        const uint32_t v = __float_as_uint(__builtin_fabsf(r[w * kWave + uint32_t(__builtin_ctzll(m))]));
        if (pass == 1) atomicAdd(&s_hist[v >> 21], 1u);
        else if (pass == 2) { if ((v >> 21) == prefix) atomicAdd(&s_hist[(v >> 10) & 2047u], 1u); }
        else if ((v >> 10) == prefix) atomicAdd(&s_hist[v & 1023u], 1u);
      }
    }
    __syncthreads();
    uint32_t d;
    if (pass == 3) find_digit<kBins3>(s_hist, rank, d, rank); else find_digit<kBins1>(s_hist, rank, d, rank);
    prefix = pass == 1 ? d : pass == 2 ? ((prefix << 11) | d) : ((prefix << 10) | d);
  }
  uint32_t at = 0, ties = rank + 1;  // of the elements equal to the value found, the first `ties` stay
#pragma unroll 1
  for (uint32_t w0 = 0; w0 < words; w0 += kSortThreads) {
    const uint32_t w = w0 + t;
    uint64_t above = 0, equal = 0;
    for (uint64_t m = w < words ? masks[w] : 0ull; m; m &= m - 1) {
      const uint64_t bit = m & (~m + 1);
      const uint32_t v = __float_as_uint(__builtin_fabsf(r[w * kWave + uint32_t(__builtin_ctzll(m))]));
      above |= v > prefix ? bit : 0ull;
      equal |= v == prefix ? bit : 0ull;
    }
    uint32_t all_equal, all_listed;
    const uint32_t equal_before = block_prefix(uint32_t(__popcll(equal)), s_wave, all_equal);
    uint32_t room = ties > equal_before ? ties - equal_before : 0u;
    uint64_t list = above;
    for (; equal && room; equal &= equal - 1, room--) list |= equal & (~equal + 1);
    uint32_t pos = at + block_prefix(uint32_t(__popcll(list)), s_wave, all_listed);
    for (; list; list &= list - 1, pos++) {
      const uint32_t e = w * kWave + uint32_t(__builtin_ctzll(list));
      const uint32_t v = __float_as_uint(r[e]);
      s_key[pos] = (v & 0x7FFFFFFFu) - thr_bits;
      s_id[pos] = e | (v & 0x80000000u);
    }
    at += all_listed;
    ties -= all_equal < ties ? all_equal : ties;
  }
  __syncthreads();
}

// The cut by one workgroup, of up to kCutKeep candidates (listed ones: kCutLds, cut_wide).  What bounds it is the chain of workgroup-wide steps, so the sort
// has as few as possible: the keys (distance of |r| above the threshold in bit patterns) go into 8192 bins by exponent
// and eight further bits of the distance as a float - fine where keys crowd just above the threshold, however far the
// largest lies (4096 bins: 0.8 and 1.2 us longer over the comparisons within them, for 1049 and 2360 kept) - the bins are laid out one after the other, and a key's place is its bin's first place plus the number
// of keys of the bin that come before it (larger, or equal with a smaller index).  Where a bin is crowded all the same
// (many equal values) the keys take a stable LSD sort by byte digits, pairs in registers between the passes and in
// LDS for the exchange.  The code is instantiated for the number of pairs per lane: unrolled for the
// most a workgroup can hold it was three times as long, and a launch of one workgroup per tensor meets a cold
// instruction cache.
constexpr uint32_t kCutBins = 8192;
constexpr uint32_t kBinWords = kCutBins / 2;   // 16 bits each: there are at most kCutLds keys
constexpr uint32_t kCutCrowd = 128;   // keys of one bin from which the digit sort is the quicker one
struct CutArgs {
  uint32_t* stage;   // LDS: 2 * kCutLds words
  uint32_t* bins;    // LDS: kBinWords + 4 words, the first kBinWords zero
  uint32_t* wave;    // LDS: a word per wave, of the cut's own
  float* r;
  uint8_t* out;
  uint32_t n, keep, thr_bits;
  bool cleared;      // r holds zeros at the candidates: the dropped ones go back.  Else their values: the kept ones are cleared
  uint32_t first, all;   // place in the message of the largest pair at hand, and entries of the message
  __device__ __forceinline__ uint32_t value(uint32_t key, uint32_t id) const { return (key + thr_bits) | (id & 0x80000000u); }
  __device__ __forceinline__ void entry(uint32_t place, uint32_t key, uint32_t id) const {   // of the message
    reinterpret_cast<uint32_t*>(out + 4)[first + place] = id & 0x7FFFFFFFu;
    reinterpret_cast<uint32_t*>(out + 4 + size_t(all) * 4)[first + place] = value(key, id);
  }
  __device__ __forceinline__ void residual(uint32_t place, uint32_t key, uint32_t id) const {
    if (cleared != (place < keep)) r[id & 0x7FFFFFFFu] = cleared ? __uint_as_float(value(key, id)) : 0.0f;
  }
  __device__ __forceinline__ void put(uint32_t place, uint32_t key, uint32_t id) const {
    if (place < keep) entry(place, key, id);
    residual(place, key, id);
  }
};

__device__ __forceinline__ uint32_t cut_bin(uint32_t key) { return kCutBins - 1 - ((__float_as_uint(float(key)) >> 15) - (127u << 8)); }
// One more at a bin's count (or its next place); what was there before.
__device__ __forceinline__ uint32_t bin_step(const CutArgs& f, uint32_t bin) {
  const uint32_t shift = (bin & 1u) * 16u;
  return (atomicAdd(&f.bins[bin >> 1], 1u << shift) >> shift) & 0xFFFFu;
}
__device__ __forceinline__ uint32_t bin_at(const CutArgs& f, uint32_t bin) { return reinterpret_cast<const uint16_t*>(f.bins)[bin]; }
// From the counts of the bins to their first places, in place (all lanes, behind the barrier that follows the counting).
// False: some bin is crowded, and the counts are still there.
__device__ __forceinline__ bool bins_laid_out(const CutArgs& f) {
  const uint32_t t = threadIdx.x;
  static_assert(kBinWords == 4 * kSortThreads && kCutLds < 65536, "four words to a lane, places of 16 bits");
  const uint4 c = reinterpret_cast<const uint4*>(f.bins)[t];
  const uint32_t word[4] = {c.x, c.y, c.z, c.w};
  uint32_t sum = 0, most = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const uint32_t a = word[k] & 0xFFFFu, b = word[k] >> 16;
    sum += a + b;
    most = a > most ? a : most;
    most = b > most ? b : most;
  }
  uint32_t total;
  bool crowded;
  uint32_t at = block_prefix_once(sum, most > kCutCrowd, f.wave, total, crowded);
  if (crowded) return false;
  uint32_t first[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const uint32_t a = word[k] & 0xFFFFu, b = word[k] >> 16;
    first[k] = at | ((at + a) << 16);
    at += a + b;
  }
  reinterpret_cast<uint4*>(f.bins)[t] = make_uint4(first[0], first[1], first[2], first[3]);
  if (t == 0) f.bins[kBinWords] = total;
  __syncthreads();
  return true;
}
template <int PER>
__device__ __forceinline__ void stage_pairs(const CutArgs& f, const uint32_t (&key)[PER], const uint32_t (&id)[PER]) {
#pragma unroll
  for (int j = 0; j < PER; j++) {
    const uint32_t x = uint32_t(j) * kSortThreads + threadIdx.x;
    if (x < f.n) { f.stage[x] = key[j]; f.stage[kCutLds + x] = id[j]; }
  }
  __syncthreads();
}

// A pair as one number, larger for what comes first: the key, then the smaller index (the sign in the last bit).
__device__ __forceinline__ uint64_t ranked(uint32_t key, uint32_t id) { return (uint64_t(key) << 32) | ~((id << 1) | (id >> 31)); }
__device__ __forceinline__ uint32_t ranked_key(uint64_t p) { return uint32_t(p >> 32); }
__device__ __forceinline__ uint32_t ranked_id(uint64_t p) { const uint32_t x = ~uint32_t(p); return (x >> 1) | (x << 31); }

// n pairs, lane t with those at t, t + 1024 ... (in ascending index order; the sign in the index's top bit).  False: some
// bin is crowded, nothing has been written, and the pairs are in LDS, [kCutLds] keys and then [kCutLds] indices.
template <int PER>
__device__ __forceinline__ bool cut_by_bins(const CutArgs& f, const uint32_t (&key)[PER], const uint32_t (&id)[PER]) {
  const uint32_t t = threadIdx.x, n = f.n;
  uint64_t* s_pair = reinterpret_cast<uint64_t*>(f.stage);
  uint32_t bin[PER], slot[PER];
#pragma unroll
  for (int j = 0; j < PER; j++) {
    const bool live = uint32_t(j) * kSortThreads + t < n;
    bin[j] = live ? cut_bin(key[j]) : 0u;
    slot[j] = live ? bin_step(f, bin[j]) : 0u;
  }
  __syncthreads();
  if (!bins_laid_out(f)) {
    stage_pairs<PER>(f, key, id);
    return false;
  }
  uint64_t own[PER];
  uint32_t lo[PER], len[PER], place[PER], longest = 0;
#pragma unroll
  for (int j = 0; j < PER; j++) {
    const bool live = uint32_t(j) * kSortThreads + t < n;
    own[j] = ranked(key[j], id[j]);
    place[j] = lo[j] = live ? bin_at(f, bin[j]) : 0u;
    len[j] = live ? bin_at(f, bin[j] + 1) - lo[j] : 0u;
    slot[j] += lo[j];
    longest = len[j] > longest ? len[j] : longest;
    if (live) s_pair[slot[j]] = own[j];
  }
  __syncthreads();
#pragma unroll 1
  for (uint32_t q = 0; q < longest; q++) {   // the lane's pairs side by side: their LDS reads overlap
    uint64_t k[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) k[j] = s_pair[q < len[j] ? lo[j] + q : slot[j]];   // (a pair is not larger than itself)
#pragma unroll
    for (int j = 0; j < PER; j++) place[j] += k[j] > own[j] ? 1u : 0u;
  }
  // The entries in order, by way of LDS behind the pairs: a lane's own go to places all over the message, a line each of the
  // indices and of the values.
  static_assert(PER * kSortThreads <= int(kCutLds) / 2, "pairs and entries side by side");
  uint64_t* s_entry = s_pair + PER * kSortThreads;
#pragma unroll
  for (int j = 0; j < PER; j++)
    if (len[j] != 0) {
      s_entry[place[j]] = own[j];
      f.residual(place[j], key[j], id[j]);
    }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < PER; j++) {
    const uint32_t x = uint32_t(j) * kSortThreads + t;
    if (x < f.keep) f.entry(x, ranked_key(s_entry[x]), ranked_id(s_entry[x]));
  }
  return true;
}

// The same for up to kCutLds pairs that lie in memory, keys and indices: walked twice, once for the counts and once into
// their bins, and then bin by bin (sixteen pairs a lane in registers, as above, spill).  Crowded bins: false, and nothing
// is left in LDS.
__device__ __forceinline__ bool cut_wide(const CutArgs& f, const uint32_t* __restrict__ keys, const uint32_t* __restrict__ cand) {
  constexpr uint32_t kAtOnce = 4;
  const uint32_t t = threadIdx.x, n = f.n;
  uint64_t* s_pair = reinterpret_cast<uint64_t*>(f.stage);
#pragma unroll 1
  for (uint32_t x0 = t; x0 < n; x0 += kAtOnce * kSortThreads) {
    uint32_t key[kAtOnce];
#pragma unroll
    for (uint32_t j = 0; j < kAtOnce; j++) key[j] = x0 + j * kSortThreads < n ? keys[x0 + j * kSortThreads] : 0u;
#pragma unroll
    for (uint32_t j = 0; j < kAtOnce; j++)
      if (x0 + j * kSortThreads < n) bin_step(f, cut_bin(key[j]));
  }
  __syncthreads();
  if (!bins_laid_out(f)) return false;
#pragma unroll 1
  for (uint32_t x0 = t; x0 < n; x0 += kAtOnce * kSortThreads) {
    uint2 pair[kAtOnce];
#pragma unroll
    for (uint32_t j = 0; j < kAtOnce; j++) {
      const uint32_t x = x0 + j * kSortThreads;
      pair[j] = x < n ? make_uint2(keys[x], cand[x]) : make_uint2(0u, 0u);
    }
#pragma unroll
    for (uint32_t j = 0; j < kAtOnce; j++)
      if (x0 + j * kSortThreads < n) s_pair[bin_step(f, cut_bin(pair[j].x))] = ranked(pair[j].x, pair[j].y);
  }
  __syncthreads();   // at a bin there is now the place behind its last pair
#pragma unroll 1
  for (uint32_t x = t; x < n; x += kSortThreads) {
    const uint64_t own = s_pair[x];
    const uint32_t b = cut_bin(ranked_key(own)), lo = b ? bin_at(f, b - 1) : 0u, hi = bin_at(f, b);
    uint32_t place = lo;
#pragma unroll 4
    for (uint32_t q = lo; q < hi; q++) place += s_pair[q] > own ? 1u : 0u;
    f.put(place, ranked_key(own), ranked_id(own));
  }
  return true;
}

// The same for many equal or nearly equal keys: the digit sort.
__device__ __forceinline__ void cut_crowded(const CutArgs& f) {
  constexpr uint32_t BINS = 256, kBinWaves = BINS / kWave;
  constexpr int kPer = int(kCutKeep) / kSortThreads;
  __shared__ uint32_t s_part[kBinWaves], s_max[kSortWaves];
  static_assert(kBinWords >= kSortWaves * BINS, "one block for both");
  uint32_t (*s_cnt)[BINS] = reinterpret_cast<uint32_t (*)[BINS]>(f.bins);
  uint32_t* s_key = f.stage;
  uint32_t* s_id = f.stage + kCutLds;
  const uint32_t t = threadIdx.x, lane = t & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(t / kWave);
  const uint32_t n = f.n;
  // pairs in order, the same number of rounds of 64 per wave for every wave
  const uint32_t per = cdiv(n, kSortThreads);
  const uint32_t x0 = wave * per * kWave + lane;
  uint32_t key[kPer], id[kPer], big = 0;
#pragma unroll
  for (int j = 0; j < kPer; j++) {
    const uint32_t x = x0 + uint32_t(j) * kWave;
    const bool live = uint32_t(j) < per && x < n;
    id[j] = live ? s_id[x] : 0u;
    key[j] = live ? s_key[x] : 0u;
    big = key[j] > big ? key[j] : big;
  }
  big = wave_max_u32(big);
  if (lane == 0) s_max[wave] = big;
  __syncthreads();   // also: every pair has been read
#pragma unroll
  for (int w = 0; w < kSortWaves; w++) big = s_max[w] > big ? s_max[w] : big;
  const int passes = big ? (39 - __builtin_clz(big)) / 8 : 1;
#pragma unroll 1
  for (int pass = 0; pass < passes; pass++) {
    const int shift = pass * 8;
#pragma unroll
    for (uint32_t q = 0; q < kBinWaves; q++) s_cnt[wave][q * kWave + lane] = 0;  // own row
    uint32_t place[kPer];
#pragma unroll
    for (int j = 0; j < kPer; j++) {
      if (uint32_t(j) < per) {
        const bool live = x0 + uint32_t(j) * kWave < n;
        const uint32_t bin = (BINS - 1) - ((key[j] >> shift) & (BINS - 1));
        const uint64_t same = match_bin<8>(bin, live);
        const uint32_t rank = uint32_t(__popcll(same & ((uint64_t(1) << lane) - 1)));
        uint32_t base = 0;
        if (live && rank == 0) {
          base = s_cnt[wave][bin];
          s_cnt[wave][bin] = base + uint32_t(__popcll(same));
        }
        base = __shfl(base, live ? __builtin_ctzll(same) : int(lane), kWave);
        place[j] = base + rank;
      }
    }
    __syncthreads();
    // bin t: the tile's total, an exclusive scan of the totals, then every wave's first place
    uint32_t c[kSortWaves], mine = 0;
    if (t < BINS) {
#pragma unroll
      for (int w = 0; w < kSortWaves; w++) { c[w] = s_cnt[w][t]; mine += c[w]; }
    }
    const uint32_t incl = wave_prefix_u32(mine);
    if (t < BINS && lane == kWave - 1) s_part[wave] = incl;
    __syncthreads();
    if (t < BINS) {
      uint32_t run = incl - mine;
      for (uint32_t w = 0; w < wave; w++) run += s_part[w];
#pragma unroll
      for (int w = 0; w < kSortWaves; w++) { s_cnt[w][t] = run; run += c[w]; }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPer; j++) {
      if (uint32_t(j) < per && x0 + uint32_t(j) * kWave < n) {
        const uint32_t p = s_cnt[wave][(BINS - 1) - ((key[j] >> shift) & (BINS - 1))] + place[j];
        s_key[p] = key[j];
        s_id[p] = id[j];
      }
    }
    __syncthreads();
    if (pass + 1 < passes) {
#pragma unroll
      for (int j = 0; j < kPer; j++) {
        const uint32_t x = x0 + uint32_t(j) * kWave;
        if (uint32_t(j) < per && x < n) { key[j] = s_key[x]; id[j] = s_id[x]; }
      }
    }
  }
#pragma unroll
  for (int j = 0; j < kPer; j++) {
    const uint32_t p = uint32_t(j) * kSortThreads + t;
    if (p < n) f.put(p, s_key[p], s_id[p]);
  }
}
// Pairs from wherever `pair(x, key, id)` finds them.
template <int PER, typename F>
__device__ __forceinline__ bool cut_loaded(const CutArgs& f, F pair) {
  uint32_t key[PER], id[PER];
#pragma unroll
  for (int j = 0; j < PER; j++) {   // (a pair beyond the last is read as the last and not used: no branch between the loads)
    const uint32_t x = uint32_t(j) * kSortThreads + threadIdx.x;
    pair(x < f.n ? x : f.n - 1, key[j], id[j]);
  }
  return cut_by_bins<PER>(f, key, id);
}

// The cut of a tensor that keeps kCutKeep entries and more, in one launch.  A workgroup takes a window of the keys, from one
// quantile of them to the next, about kWindow pairs: the windows' bounds come from kWindowSample of the keys, one out of so
// many, which a wave for each bound ranks; then it reads all the keys, counts those above its window, which is the
// place of its largest in the message, collects its own in LDS and places them as a workgroup does that has them all.  What
// bounds it is instructions, of that walk over all keys by each and of the largest window (138 thousand 26 us with windows of
// 1024 pairs on average, 31 with 1536; 10 thousand 11.8).  The digit sort's six launches took 44 and more: us per
// encode with a cut, sort -> windows, 10 thousand kept of 1 M 62.6 -> 44.5 and of 10 M 92 -> 74.5, 20 thousand 119.5 -> 102,
// 60 thousand 201 -> 184, 120 thousand 104 -> 91 (12 M), 138 thousand 361 -> 345, 200 thousand 137.5 -> 127; 400 thousand
// 205 -> 233, which is why kOrderMax lies between; bf16 values 62.6 -> 51 (1 M) and 366 -> 351 (138 M).
// A value that thousands share is several quantiles, and the windows between two of these share its candidates by their places
// (order_ties).  What does not fit all the same - the sample is one of many, and one wave may read most of a window - goes part
// by part (next_part).  So all of it is settled here, and the host, which queues the launch, does not wait for it.  us per encode of
// tensors with zeros around their candidates, sort -> windows: 100 thousand candidates 107 -> 77, with a tenth of them equal 112 -> 78,
// all of them 99 -> 74; 16 thousand with six in ten equal 103 -> 74; 220 thousand with the last three in ten equal 209 -> 184; the
// largest of 220 thousand where one wave reads 115 -> 117.  (Windows that left such tensors to a sort queued behind them, the host waiting
// for their word: 127, 118, 119, 248 and 153; and 60 instead of 20 until the call returned.)  Part by part is no more than a way out:
// 100 thousand candidates laid around the sample, on purpose, so that one window has nearly all: 1.4 ms.
constexpr uint32_t kWindow = 1024, kWindowSample = 512;
constexpr uint32_t kShared = 2;   // windows that share a value; if there were fewer of them, it goes with the window above (one by
                                  // itself walked all the keys for it: 200 thousand candidates of 64 values 141 us per encode, now 93; sort 103)
constexpr uint32_t kOrderMax = 224 * 1024;   // candidates of one tensor; for all of a call: windows_pay
// False: a bin is crowded (many equal keys), nothing has been written, and the pairs are in LDS as cut_crowded takes them, in the
// order of the candidates.  That order comes from bins of the places among those, so wide that no more than kWideBin can share one.
template <int PER>
__device__ __forceinline__ bool window_by_bins(const CutArgs& f, uint32_t below, const uint32_t* s_found,
                                               const uint32_t* __restrict__ keys, const int32_t* __restrict__ ids) {
  constexpr uint32_t kWideBin = (kOrderMax + kCutBins - 1) / kCutBins;
  static_assert(kWideBin <= kCutCrowd, "no bin of places is crowded");
  const uint32_t t = threadIdx.x;
  uint32_t key[PER], id[PER], at[PER];
#pragma unroll
  for (int j = 0; j < PER; j++) {
    const uint32_t x = uint32_t(j) * kSortThreads + t;
    at[j] = s_found[x < f.n ? x : f.n - 1];
    key[j] = keys[at[j]] - below;
    id[j] = uint32_t(ids[at[j]]);
  }
  if (cut_by_bins<PER>(f, key, id)) return true;
  reinterpret_cast<uint4*>(f.bins)[t] = make_uint4(0, 0, 0, 0);
  __syncthreads();
  uint32_t slot[PER];
#pragma unroll
  for (int j = 0; j < PER; j++) slot[j] = uint32_t(j) * kSortThreads + t < f.n ? bin_step(f, at[j] / kWideBin) : 0u;
  __syncthreads();
  bins_laid_out(f);
  uint32_t* s_at = f.stage + kCutLds + kCutKeep;
#pragma unroll
  for (int j = 0; j < PER; j++)
    if (uint32_t(j) * kSortThreads + t < f.n) s_at[bin_at(f, at[j] / kWideBin) + slot[j]] = at[j];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < PER; j++) {
    if (uint32_t(j) * kSortThreads + t >= f.n) continue;
    const uint32_t lo = bin_at(f, at[j] / kWideBin), hi = bin_at(f, at[j] / kWideBin + 1);
    uint32_t place = lo;
#pragma unroll 1
    for (uint32_t q = lo; q < hi; q++) place += s_at[q] < at[j] ? 1u : 0u;
    f.stage[place] = key[j];
    f.stage[kCutLds + place] = id[j];
  }
  __syncthreads();
  return false;
}
// The candidates whose key is `v`, of the part-th of `parts` stretches of the keys, in their order to their places in the message.
// (`f`: with all of the message's entries.)  Gives how many candidates come before the stretch's first and how many there are.
__device__ __forceinline__ void order_ties(const CutArgs& f, const uint32_t* __restrict__ keys, const int32_t* __restrict__ ids, uint32_t v,
                                           uint32_t part, uint32_t parts, uint32_t& before, uint32_t& found) {
  const uint32_t t = threadIdx.x, quads = (f.n + 3) / 4;
  const uint32_t from = quads * part / parts, to = quads * (part + 1) / parts;
  const uint4* __restrict__ quad = reinterpret_cast<const uint4*>(keys);
  auto take = [&](uint32_t q, uint32_t (&k)[4]) {   // zeros behind the last one: no key is
    const uint4 x = quad[q];
    k[0] = x.x; k[1] = x.y; k[2] = x.z; k[3] = x.w;
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) k[i] = 4 * q + i < f.n ? k[i] : 0u;
  };
  uint32_t mine = 0;
#pragma unroll 4
  for (uint32_t q = t; q < quads; q += kSortThreads) {
    uint32_t k[4];
    take(q, k);
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) mine += k[i] > v || (q < from && k[i] == v) ? 1u : 0u;
  }
  found = 0;
  block_prefix(mine, f.wave, before);
  // Four quads to a lane of a stretch that has so many (one: 57 us for 200 thousand keys in one stretch, each round waits for its keys).
  constexpr uint32_t kAtOnce = 4;
  const uint32_t per = cdiv(to - from, kSortThreads) < kAtOnce ? cdiv(to - from, kSortThreads) : kAtOnce;
#pragma unroll 1
  for (uint32_t q0 = from; q0 < to && before + found < f.keep; q0 += per * kSortThreads) {
    const uint32_t q = q0 + per * t;
    uint32_t marks = 0;
#pragma unroll
    for (uint32_t j = 0; j < kAtOnce; j++) {
      const bool in = j < per && q + j < to;
      uint32_t k[4];
      take(in ? q + j : from, k);
#pragma unroll
      for (uint32_t i = 0; i < 4; i++) marks |= in && k[i] == v ? 1u << (4 * j + i) : 0u;
    }
    uint32_t all;
    uint32_t place = before + found + block_prefix(uint32_t(__builtin_popcount(marks)), f.wave, all);
    for (; marks != 0; marks &= marks - 1) f.put(place++, v, uint32_t(ids[4 * q + uint32_t(__builtin_ctz(marks))]));
    found += all;
  }
}
// Of the `left` keys in [lo, top), the largest, kPart of them at most: where they lie to s_found, how many of them there are as the
// result (0: none are left), the least key that is theirs to `bottom`.  Where not all of them fit: bins of 1 << shift keys each,
// larger ones first, as many from the front as hold no more than fit; if the first one does not, its keys in finer ones, down to
// one value, whose candidates go to the message at once.
constexpr uint32_t kPart = 4096;
__device__ __forceinline__ uint32_t next_part(const CutArgs& f, const uint32_t* __restrict__ keys, const int32_t* __restrict__ ids, uint32_t lo,
                                              uint32_t& top, uint32_t& bottom, uint32_t& first, uint32_t& left, uint32_t* s_found,
                                              uint32_t* s_cut) {
  const uint32_t t = threadIdx.x;
  auto walk = [&](auto key_at) {   // (a place behind the last key: zero, below all that is asked for)
    const uint4* __restrict__ quad = reinterpret_cast<const uint4*>(keys);
    const uint32_t quads = (f.n + 3) / 4;
#pragma unroll 4
    for (uint32_t q = t; q < quads; q += kSortThreads) {
      const uint4 x = quad[q];
      const uint32_t k[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
      for (uint32_t i = 0; i < 4; i++) key_at(4 * q + i < f.n ? k[i] : 0u, 4 * q + i);
    }
  };
  bottom = lo;
#pragma unroll 1
  while (left > 0 && first < f.keep) {
    uint32_t count = left;
    if (t == 0) s_cut[2] = 0;
    if (left > kPart) {
      const uint32_t span = top - bottom, wide = 32 - uint32_t(__builtin_clz(span)), shift = wide > 12 ? wide - 12 : 0u;
      static_assert(kBinWords == 1u << 12 && kBinWords == 4 * kSortThreads, "four bins to a lane");
      reinterpret_cast<uint4*>(f.bins)[t] = make_uint4(0, 0, 0, 0);
      __syncthreads();
      walk([&](uint32_t k, uint32_t) {
        const uint32_t d = top - 1 - k;
        if (d < span) atomicAdd(&f.bins[d >> shift], 1u);
      });
      __syncthreads();
      const uint4 c = reinterpret_cast<const uint4*>(f.bins)[t];
      const uint32_t bin[4] = {c.x, c.y, c.z, c.w};
      uint32_t total;
      uint32_t at = block_prefix(c.x + c.y + c.z + c.w, f.wave, total);
      if (t == 0) { s_cut[0] = kBinWords; s_cut[1] = total; }
      __syncthreads();
#pragma unroll
      for (uint32_t i = 0; i < 4; i++) {   // the bin that no longer fits, if there is one, and how many keys lie before it
        if (at <= kPart && at + bin[i] > kPart) { s_cut[0] = 4 * t + i; s_cut[1] = at; }
        at += bin[i];
      }
      __syncthreads();
      const uint32_t bins = s_cut[0];
      count = s_cut[1];
      if (bins == 0 && shift > 0) {
        bottom = top - (1u << shift);   // there are more bins than that one
        continue;
      }
      if (bins == 0) {
        uint32_t before, found;
        order_ties(f, keys, ids, top - 1, 0, 1, before, found);
        first += found;   // (not all of them where the message ends there)
        left -= found;
        top -= 1;
        bottom = lo;
        continue;
      }
      if (bins < kBinWords) bottom = top - (bins << shift);
      if (count == 0) {
        top = bottom;
        bottom = lo;
        continue;
      }
    }
    reinterpret_cast<uint4*>(f.bins)[t] = make_uint4(0, 0, 0, 0);
    __syncthreads();
    walk([&](uint32_t k, uint32_t x) {
      if (k >= bottom && k < top) s_found[atomicAdd(&s_cut[2], 1u)] = x;
    });
    __syncthreads();
    return count;
  }
  return 0;
}
template <int CAP>
__global__ __launch_bounds__(kSortThreads) void gd_order_kernel(const SortArgs<CAP> a) {
  // (Aligned by name: behind an odd number of words the pairs' 64-bit accesses took this launch from 27 to 42 us.)
  extern __shared__ __align__(16) uint32_t s_stage[];   // 2 * kCutLds words: where the window's keys lie, a list per wave and then all of them; the pairs
  __shared__ __align__(16) uint32_t s_bins[kBinWords + 4];
  __shared__ uint32_t s_wave[kSortWaves], s_cut_wave[kSortWaves], s_bound[3], s_cut[3];
  const uint32_t t = threadIdx.x, lane = t & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(t / kWave);
  const int s = find_segment<CAP>(a.tile_start, a.nseg, blockIdx.x);
  const SortSeg& sg = a.seg[s];
  const uint32_t window = uint32_t(int(blockIdx.x) - a.tile_start[s]), windows = uint32_t(a.tile_start[s + 1] - a.tile_start[s]);
  const CutLayout cl = cut_layout(sg.cap);
  const uint32_t* __restrict__ keys = sort_keys(sg, cl, 0);
  const uint32_t n = sg.n, keep = sg.keep;
  const int32_t* __restrict__ ids = sort_ids(sg, cl, 0);
  constexpr uint32_t kOwn = kWindowSample / kWave;
  auto sample = [&](uint32_t (&key)[kOwn]) {   // one of each stretch, anywhere in it: no regular order of the values passes between them
#pragma unroll
    for (uint32_t j = 0; j < kOwn; j++) {
      const uint32_t x = j * kWave + lane;
      key[j] = keys[uint32_t(uint64_t(x) * n / kWindowSample) + (((x * 0x9E3779B1u) >> 16) * (n / kWindowSample) >> 16)];
    }
  };
  reinterpret_cast<uint4*>(s_bins)[t] = make_uint4(0, 0, 0, 0);
  // The last window bound that a value reaches: those between its first one and that one are its own.
  auto last_bound = [&](const uint32_t (&key)[kOwn], uint32_t v) {
    uint32_t reach = 0;
#pragma unroll
    for (uint32_t j = 0; j < kOwn; j++) reach += uint32_t(__popcll(__ballot(key[j] >= v)));
    const uint32_t to = cdiv(reach * windows, kWindowSample) - 1;
    return v == 1u ? windows : to < windows - 1 ? to : windows - 1;
  };
  if (wave < 3) {   // one for each bound, and one looks how far the lower one reaches (the others too: 4 us more, a request for each of their keys)
    uint32_t key[kOwn];
    sample(key);
    const uint32_t w = window + (wave > 0 ? 1u : 0u);
    uint32_t bound = w == 0 ? 0xFFFFFFFFu : 1u;   // keys are at least 1
    if (w > 0 && w < windows) {
      bound = wave_rank<int(kOwn), 0>(key, uint32_t(uint64_t(w) * kWindowSample / windows), 0u);
      bound = bound > 1u ? bound : 1u;
    }
    if (wave == 2) bound = last_bound(key, bound);
    if (lane == 0) s_bound[wave] = bound;
  }
  __syncthreads();
  const uint32_t hi = s_bound[0];
  uint32_t lo = s_bound[1];
  if (window == 0 && t == 0) *reinterpret_cast<int32_t*>(sg.msg) = int32_t(4 + keep * 8);
  const CutArgs whole{s_stage, s_bins, s_wave, sg.r, sg.msg, n, keep, sg.thr_bits, false, 0, keep};
  if (hi == lo) {   // its quantiles are one value
    uint32_t key[kOwn], above = 0;
    sample(key);
#pragma unroll
    for (uint32_t j = 0; j < kOwn; j++) above += uint32_t(__popcll(__ballot(key[j] > lo)));
    uint32_t from = cdiv(above * windows, kWindowSample);
    from = from > 1u ? from : 1u;
    const uint32_t to = s_bound[2];
    uint32_t before, found;
    if (to - from >= kShared) order_ties(whole, keys, ids, lo, window - from, to - from, before, found);
    return;
  }
  if (s_bound[2] - (window + 1) >= kShared) {   // the windows below see to that value
    lo++;
    if (hi == lo) return;
  }
  // A lane marks those of its sixteen keys that are in the window, and the wave then lists the marked ones, one of each lane at
  // a time: no branch on the way (with one at every key the walk over 138 thousand took 20 us).
  constexpr uint32_t kListOf = kCutLds / kSortWaves;   // a wave's list, next to sixteen times what it finds on average
  uint32_t* s_list = s_stage + wave * kListOf;
  uint32_t above = 0, mine = 0;                         // of the wave
  constexpr uint32_t kAtOnce = 4;
  const uint4* __restrict__ quads = reinterpret_cast<const uint4*>(keys);
  const uint32_t last = (n - 1) / 4, span = hi - lo;
#pragma unroll 1
  for (uint32_t q0 = 0; q0 <= last; q0 += kAtOnce * kSortThreads) {
    uint4 k[kAtOnce];
    uint32_t marks = 0;
#pragma unroll
    for (uint32_t j = 0; j < kAtOnce; j++) {
      const uint32_t q = q0 + j * kSortThreads + t;
      k[j] = quads[q < last ? q : last];
    }
    const bool ends = q0 + kAtOnce * kSortThreads > last;   // uniform
#pragma unroll
    for (uint32_t j = 0; j < kAtOnce; j++) {
      const uint32_t x = 4 * (q0 + j * kSortThreads + t);
      uint32_t v[4] = {k[j].x, k[j].y, k[j].z, k[j].w};
      if (ends) {   // zeros are below every window
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) v[i] = x + i < n ? v[i] : 0u;
      }
#pragma unroll
      for (uint32_t i = 0; i < 4; i++) {
        above += uint32_t(__popcll(__ballot(v[i] >= hi)));
        marks |= v[i] - lo < span ? 1u << (4 * j + i) : 0u;
      }
    }
#pragma unroll 1
    for (uint64_t some = __ballot(marks != 0); some != 0; some = __ballot(marks != 0)) {
      const uint32_t at = mine + __builtin_amdgcn_mbcnt_hi(uint32_t(some >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(some), 0u));
      const uint32_t i = marks ? uint32_t(__builtin_ctz(marks)) : 0u;
      if (marks != 0 && at < kListOf) s_list[at] = 4 * (q0 + i / 4 * kSortThreads + t) + i % 4;
      marks &= marks - 1;   // 0 stays 0
      mine += uint32_t(__popcll(some));
    }
  }
  if (lane == 0) { s_wave[wave] = above; s_cut_wave[wave] = mine; }
  __syncthreads();
  uint32_t first, found;
  before_wave(s_wave[lane & 15], first);
  const uint32_t in_wave = s_cut_wave[lane & 15], start = before_wave(in_wave, found);
  const bool fits = __ballot(in_wave > kListOf) == 0 && found <= kCutKeep;
  if (found == 0 || first >= keep) return;   // nothing of it is sent
  uint32_t* s_found = s_stage + kCutLds;
  auto pairs = [&](uint32_t below, uint32_t count) {
    const uint32_t kept = keep - first < count ? keep - first : count;
    return CutArgs{s_stage, s_bins, s_cut_wave, sg.r, sg.msg, count, kept, sg.thr_bits + below, false, first, keep};
  };
  if (fits) {
    for (uint32_t i = lane; i < mine; i += kWave) s_found[start + i] = s_list[i];
    __syncthreads();
    const uint32_t below = lo - 1;
    const CutArgs f = pairs(below, found);
    const bool done = found <= 2 * kSortThreads   ? window_by_bins<2>(f, below, s_found, keys, ids)
                      : found <= 3 * kSortThreads ? window_by_bins<3>(f, below, s_found, keys, ids)
                      : found <= 4 * kSortThreads ? window_by_bins<4>(f, below, s_found, keys, ids)
                                                  : window_by_bins<8>(f, below, s_found, keys, ids);
    if (!done) cut_crowded(f);
    return;
  }
  uint32_t top = hi, bottom;
#pragma unroll 1
  for (;;) {
    __syncthreads();
    const uint32_t count = next_part(whole, keys, ids, lo, top, bottom, first, found, s_found, s_cut);
    if (count == 0) return;
    const CutArgs f = pairs(bottom - 1, count);
    if (!window_by_bins<int(kPart) / kSortThreads>(f, bottom - 1, s_found, keys, ids)) cut_crowded(f);
    first += count;
    found -= count;
    top = bottom;
  }
}

// What is left to do for a tensor that keeps at most kFinishKeep entries once the pass has marked its candidates,
// by one workgroup in one launch: list them, cut them if there are too many, write the message and clear the
// residual.  (Beyond that the values' random reads and the clearing's random writes, at about 700 lines a
// microsecond for one CU, take longer than the expand launch that spreads them.)  A group of lanes looks after a tile
// (as many as give every lane something to do), a lane after a run of the tile's mask words, of which the tile's coarse
// word names the few that have a bit set; lanes in order, so one prefix over the workgroup's counts puts the indices
// in ascending order in LDS.
// One tensor of 1 M: scan, expand and the cut's seven launches 36 us with the host's turn-around -> 6.1 us on average;
// ResNet-50's 161 tensors 58 -> 10.3 us.  What bounds it is instructions (before_wave) and lines (list_room): from the kernel's
// start, us, for a cut of 2481 to 2360, lengths 1.6, their prefix 2.1, places in LDS 3.9, entries 6.3, counted into bins 6.6, laid out
// 8.0, compared 9.5, written 11 (before: 1.8, 2.5, 4.5, 6.7, 7.5, 9.2, 12.5, 14.5); a cut of 1230 to 1049 8 (before 10).
// Larger ones that still fit are only cut here, behind the expand launch.  All of it is queued before the host knows any
// count.
// The cut of the tensors that keep between kFinishKeep and kCutKeep entries, whose candidates and keys the expand
// launch has listed (or, where they are too many for the list or for LDS, are found again in the mask).
__device__ __forceinline__ void cut_listed(const GdSeg& sg, uint32_t* s_stage, uint32_t* s_bins, uint32_t* s_wave, uint32_t* s_cut_wave) {
  const uint32_t found = seg_state(sg)->total, keep = sg.limit, thr_bits = seg_state(sg)->thr_bits;
  if (found <= keep) return;
  const uint32_t t = threadIdx.x;
  if (t == 0) *reinterpret_cast<int32_t*>(sg.out) = int32_t(4 + keep * 8);
  if (keep == 0) return;
  const CutLayout cl = cut_layout(sg.cap);
  const uint32_t* __restrict__ keys = reinterpret_cast<const uint32_t*>(sg.cut + cl.ka);
  const uint32_t* __restrict__ cand = reinterpret_cast<const uint32_t*>(sg.cut + cl.ia);
  auto clear_bins = [&]() {
    reinterpret_cast<uint4*>(s_bins)[t] = make_uint4(0, 0, 0, 0);
    __syncthreads();
  };
  if (found <= sg.cap && found > kCutKeep && found <= kCutLds) {
    clear_bins();
    if (cut_wide(CutArgs{s_stage, s_bins, s_cut_wave, sg.r, sg.out, found, keep, thr_bits, false, 0, keep}, keys, cand)) return;
    __syncthreads();
  }
  const bool listed = found <= sg.cap && found <= kCutKeep;
  if (!listed) {
    const GdLayout l = gd_layout(sg.n, sg.sample_cnt);
    top_of_masks(reinterpret_cast<const uint64_t*>(sg.ws + l.masks), sg.r, sg.n, keep, thr_bits, s_bins, s_wave, s_stage, s_stage + kCutLds);
  }
  clear_bins();
  const CutArgs f{s_stage, s_bins, s_cut_wave, sg.r, sg.out, listed ? found : keep, keep, thr_bits, false, 0, keep};
  bool done;
  if (listed) {
    auto pair = [=](uint32_t x, uint32_t& key, uint32_t& id) { key = keys[x]; id = cand[x]; };
    done = f.n <= 2 * kSortThreads ? cut_loaded<2>(f, pair) : f.n <= 4 * kSortThreads ? cut_loaded<4>(f, pair) : cut_loaded<8>(f, pair);
  } else {
    done = cut_loaded<8>(f, [=](uint32_t x, uint32_t& key, uint32_t& id) { key = f.stage[x]; id = f.stage[kCutLds + x]; });
  }
  if (!done) cut_crowded(f);
}

template <int CAP>
__global__ __launch_bounds__(kSortThreads) void gd_finish_kernel(const GdArgs<CAP> a) {
  extern __shared__ __align__(16) uint32_t s_stage[];          // [kCutLds] keys, then [kCutLds] indices; or pairs of them
  __shared__ __align__(16) uint32_t s_bins[kBinWords + 4];   // counts, then first places; the rank search's histogram; the digit sort's counts
  __shared__ uint32_t s_wave[kSortWaves], s_cut_wave[kSortWaves];
  static_assert(kBinWords >= uint32_t(kBins1), "one block for both");
  uint32_t* s_key = s_stage;
  uint32_t* s_id = s_stage + kCutLds;
  const GdSeg& sg = a.seg[find_segment<CAP>(a.tile_start, a.nseg, blockIdx.x)];
  if (!one_workgroup(sg.n, sg.limit)) {
    cut_listed(sg, s_stage, s_bins, s_wave, s_cut_wave);
    return;
  }
  const GdLayout l = gd_layout(sg.n, sg.sample_cnt);
  const uint64_t* __restrict__ masks = reinterpret_cast<const uint64_t*>(sg.ws + l.masks);
  const uint64_t* __restrict__ coarse = reinterpret_cast<const uint64_t*>(sg.ws + l.coarse);
  const uint32_t thr_bits = seg_state(sg)->thr_bits, keep = sg.limit;
  const uint32_t t = threadIdx.x;
  const uint32_t ntiles = cdiv(sg.n, kTile);
  float* __restrict__ r = sg.r;

  // The pass's own lists, a few of them to a lane: where each entry of the tensor's list of candidates lies, and then the
  // entries, each a load that depends on nothing but its place.  (Through the masks every candidate is a word of the mask and
  // then a line of r.  Each list's first entries requested along with its length, six to a lane: as many requests as there are
  // lists, times three, which one CU takes 3 us over for 2304 of them.)
  const uint32_t room = list_room(sg.n, keep);
  const bool cleared = a.residual != 0 && clears_listed(sg.n, keep);
  uint2* entries = reinterpret_cast<uint2*>(sg.ws + l.hitlist);   // what has no room in the lists, from `lists0` on the lists
  const uint2* __restrict__ list = seg_list(sg, l);
  const uint32_t lists0 = uint32_t((l.end - l.hitlist) / sizeof(uint2));   // (below 2^31 at any size of sample)
  static_assert(sizeof(uint32_t) * kHitExtra >= sizeof(uint2) * kCutKeep, "which the provisional path's block holds");
  uint32_t n = 0, pos = 0;
  reinterpret_cast<uint4*>(s_bins)[t] = make_uint4(0, 0, 0, 0);
  if (room != 0) {
    constexpr uint32_t kAtOnce = 4;
    const uint32_t nlists = ntiles * (kThreads / kWave), per = cdiv(nlists, kSortThreads), first = t * per;
    const uint16_t* __restrict__ lengths = reinterpret_cast<const uint16_t*>(sg.ws + l.wcnt);
    uint32_t c[kAtOnce], mine = 0;
    bool over = false;
    auto take = [&](uint32_t q0) {
#pragma unroll
      for (uint32_t q = 0; q < kAtOnce; q++) c[q] = q0 + q < per && first + q0 + q < nlists ? lengths[first + q0 + q] : 0u;
    };
    for (uint32_t q0 = 0; q0 < per; q0 += kAtOnce) {
      take(q0);
#pragma unroll
      for (uint32_t q = 0; q < kAtOnce; q++) { mine += c[q]; over = over || c[q] > room; }
    }
    bool some_over;
    pos = block_prefix_once(mine, over, s_wave, n, some_over);
    if (n <= kCutKeep) {
      if (!some_over) {
        for (uint32_t q0 = 0; q0 < per; q0 += kAtOnce) {
          if (per > kAtOnce) take(q0);
#pragma unroll
          for (uint32_t q = 0; q < kAtOnce; q++)
            for (uint32_t j = 0; j < c[q]; j++) s_id[pos++] = lists0 + (first + q0 + q) * room + j;
        }
      } else {
        // What has no room in its list the masks name; its values get places in a block that is free here.  (All candidates through the masks as soon as
        // one list is too short: one million, half of its large values within 1 in 1500, 60 us per encode, now 34; 2.4 M with 37
        // lists of 2400 too short by four 59, and 65 with what the pass had cleared put back first, now 55; with 146 such lists 53, now 49.)
        for (uint32_t q = first; q < first + per && q < nlists; q++) {
          const uint32_t found = lengths[q];
          for (uint32_t j = 0; j < found && j < room; j++) s_id[pos + j] = lists0 + q * room + j;
          pos += found;
        }
        uint32_t start = pos - mine;
        // by their element and a mark; a row of lanes to a list, a word of the mask to a lane
        static_assert(kWaveTile / kWave == 16, "a row of words");
        const uint32_t lane = t & (kWave - 1), row = lane / 16;
#pragma unroll 1
        for (uint32_t q = first; q < first + per; q++) {
          const uint32_t found = q < nlists ? lengths[q] : 0u;
#pragma unroll 1
          for (uint64_t some = __ballot(found > room); some != 0;) {
            uint32_t of = kWave;   // whose list it is
#pragma unroll
            for (uint32_t k = 0; k < 4; k++) {
              if (row == k && some != 0) of = uint32_t(__builtin_ctzll(some));
              some &= some - 1;   // 0 stays 0
            }
            const uint32_t which = __shfl(q, int(of), kWave), at = __shfl(start, int(of), kWave);
            const uint64_t m = of < uint32_t(kWave) ? masks[size_t(which) * 16 + lane % 16] : 0ull;
            const uint32_t c = uint32_t(__popcll(m));
            uint32_t before = row_prefix_u32(c) - c;
            for (uint64_t x = m; x; x &= x - 1, before++)
              if (before >= room) s_id[at + before] = 0x80000000u | (which * uint32_t(kWaveTile) + lane % 16 * kWave + uint32_t(__builtin_ctzll(x)));
          }
          start += found;
        }
        __syncthreads();
        for (uint32_t x = t; x < n; x += kSortThreads) {
          if (!(s_id[x] >> 31)) continue;
          const uint32_t i = s_id[x] & 0x7FFFFFFFu;
          entries[x] = make_uint2(i, __float_as_uint(r[i]));
          if (cleared) r[i] = 0.0f;
          s_id[x] = x;
        }
      }
      if (t == 0) *reinterpret_cast<int32_t*>(sg.out) = int32_t(4 + (n > keep ? keep : n) * 8);
      if (n == 0 || keep == 0) return;
      __syncthreads();
      if (n <= keep) {   // gd_body.h:193-229
        int32_t* __restrict__ idx = reinterpret_cast<int32_t*>(sg.out + 4);
        uint32_t* __restrict__ val = reinterpret_cast<uint32_t*>(sg.out + 4 + size_t(n) * 4);
        for (uint32_t x0 = t; x0 < n; x0 += 3 * kSortThreads) {   // three in flight per lane
          uint2 e[3];
#pragma unroll
          for (uint32_t j = 0; j < 3; j++) e[j] = entries[s_id[x0 + j * kSortThreads < n ? x0 + j * kSortThreads : x0]];
#pragma unroll
          for (uint32_t j = 0; j < 3; j++) {
            const uint32_t x = x0 + j * kSortThreads;
            if (x < n) {
              idx[x] = int32_t(e[j].x);
              val[x] = e[j].y;
              if (!cleared) r[e[j].x] = 0.0f;
            }
          }
        }
        return;
      }
      const CutArgs f{s_stage, s_bins, s_cut_wave, r, sg.out, n, keep, thr_bits, cleared, 0, keep};
      auto pair = [=](uint32_t x, uint32_t& key, uint32_t& id) {
        const uint2 e = entries[s_id[x]];
        key = (e.y & 0x7FFFFFFFu) - thr_bits;
        id = e.x | (e.y & 0x80000000u);
      };
      const bool done = n <= kSortThreads       ? cut_loaded<1>(f, pair)
                        : n <= 2 * kSortThreads ? cut_loaded<2>(f, pair)
                        : n <= 3 * kSortThreads ? cut_loaded<3>(f, pair)
                                                : cut_loaded<8>(f, pair);
      if (!done) cut_crowded(f);
      return;
    }
    // Too many for the workgroup: the masks name them, and their values are looked up in r.  (8500 to 16 thousand candidates of a million that
    // keeps 1049 146 to 182 us per encode; 148 to 176 when the pass cleared nothing.)
    if (cleared) {
      for (uint32_t q = first; q < first + per && q < nlists; q++) {
        const uint32_t in_list = lengths[q] < room ? lengths[q] : room;
        for (uint32_t j = 0; j < in_list; j++) {
          const uint2 e = list[size_t(q) * room + j];
          r[e.x] = __uint_as_float(e.y);
        }
      }
    }
    __syncthreads();
  }

  // lanes per tile (a power of two, at most one per mask word), or tiles per lane
  int group = 0;   // log2
  while (group < 6 && (ntiles << (group + 1)) <= uint32_t(kSortThreads)) group++;
  const uint32_t per_lane = cdiv(ntiles, kSortThreads);   // 1 unless there are more tiles than lanes
  const uint32_t tile0 = group ? t >> group : t * per_lane;
  const uint32_t words = kWave >> group, word0 = (t & ((1u << group) - 1)) * words;
  const uint64_t range = words == 64 ? ~0ull : ((1ull << words) - 1) << word0;
  // The lane's words of its first tile, the first four of them in registers.
  auto four = [&](uint32_t tile, uint64_t& c, uint32_t (&e)[4], uint64_t (&m)[4]) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const uint32_t w = c ? uint32_t(__builtin_ctzll(c)) : 0u;
      e[k] = tile * uint32_t(kTile) + w * kWave;
      m[k] = c ? masks[size_t(tile) * kWave + w] : 0ull;
      c &= c - 1;   // 0 stays 0
    }
  };
  uint64_t c0 = tile0 < ntiles ? coarse[tile0] & range : 0ull, m0[4];
  uint32_t e0[4];
  four(tile0, c0, e0, m0);
  uint32_t mine = 0;
  if (group == 0) {   // whole tiles: the pass has left their counts
    for (uint32_t q = 0; q < per_lane && tile0 + q < ntiles; q++) mine += reinterpret_cast<const uint32_t*>(sg.ws + l.cnt)[tile0 + q];
  } else {
#pragma unroll
    for (int k = 0; k < 4; k++) mine += uint32_t(__popcll(m0[k]));
    for (uint64_t c = c0; c; c &= c - 1) mine += uint32_t(__popcll(masks[size_t(tile0) * kWave + uint32_t(__builtin_ctzll(c))]));
  }
  pos = block_prefix(mine, s_wave, n);
  const bool cut = n > keep;
  if (t == 0) *reinterpret_cast<int32_t*>(sg.out) = int32_t(4 + (cut ? keep : n) * 8);
  if (n == 0 || keep == 0) return;
  if (n <= kCutKeep) {
    auto list = [&](const uint32_t (&e)[4], const uint64_t (&m)[4]) {
#pragma unroll
      for (int k = 0; k < 4; k++)
        for (uint64_t x = m[k]; x; x &= x - 1, pos++) s_id[pos] = e[k] + uint32_t(__builtin_ctzll(x));
    };
    list(e0, m0);
    for (uint32_t q = 0;;) {
      while (c0) {
        four(tile0 + q, c0, e0, m0);
        list(e0, m0);
      }
      if (++q >= per_lane || tile0 + q >= ntiles) break;
      c0 = coarse[tile0 + q];
    }
    __syncthreads();
  } else {
    top_of_masks(masks, r, sg.n, keep, thr_bits, s_bins, s_wave, s_key, s_id);
    reinterpret_cast<uint4*>(s_bins)[t] = make_uint4(0, 0, 0, 0);
    n = keep;
  }
  if (!cut) {   // gd_body.h:193-229
    int32_t* __restrict__ idx = reinterpret_cast<int32_t*>(sg.out + 4);
    float* __restrict__ val = reinterpret_cast<float*>(sg.out + 4 + size_t(n) * 4);
    for (uint32_t x0 = t; x0 < n; x0 += 3 * kSortThreads) {   // three values in flight per lane
      uint32_t i[3];
      float v[3];
#pragma unroll
      for (uint32_t j = 0; j < 3; j++) i[j] = s_id[x0 + j * kSortThreads < n ? x0 + j * kSortThreads : x0];
#pragma unroll
      for (uint32_t j = 0; j < 3; j++) v[j] = r[i[j]];
#pragma unroll
      for (uint32_t j = 0; j < 3; j++) {
        const uint32_t x = x0 + j * kSortThreads;
        if (x < n) {
          idx[x] = int32_t(i[j]);
          val[x] = v[j];
          r[i[j]] = 0.0f;
        }
      }
    }
    return;
  }
  const CutArgs f{s_stage, s_bins, s_cut_wave, r, sg.out, n, keep, thr_bits, false, 0, keep};
  auto pair = [=](uint32_t x, uint32_t& key, uint32_t& id) {
    id = s_id[x];
    const uint32_t v = __float_as_uint(r[id & 0x7FFFFFFFu]);
    key = (v & 0x7FFFFFFFu) - thr_bits;
    id |= v & 0x80000000u;
  };
  const bool done = n <= kSortThreads ? cut_loaded<1>(f, pair) : n <= 3 * kSortThreads ? cut_loaded<3>(f, pair) : cut_loaded<8>(f, pair);
  if (!done) cut_crowded(f);
}

// ---- decode -----------------------------------------------------------------
// A call's messages travel as a table in the kernel arguments.  The reference reads every header on the host before
// it touches an output (gd_body.h:301-325).  Here the check runs on the device: a launch either checks all headers of
// its table itself (every workgroup reads them, one per lane - a few hundred bytes out of the L2) and leaves
// everything alone if one is bad, or has been queued after the host has seen the verdict.  The verdict is one
// 64-bit pinned word, written as soon as the first launch runs; the host polls it.
// Before, every header was a copy of its own and every message a launch or two: decoding 161 messages cost 600 us of
// an encode + decode pass of 864, now one launch of 5.
struct GdMsg {   // 32 bytes
  const uint8_t* in;
  float* out;
  uint32_t out_n;
  int32_t in_size;
  int32_t add;
  int32_t pad;
};
template <int CAP>
struct GdDecArgs {
  int32_t nseg;
  int32_t check;                // 1: check the headers of this table before anything is written
  int32_t tile_start[CAP + 1];
  GdMsg seg[CAP];
  unsigned long long* report;   // pinned: the verdict of this table's check goes here (null: nobody waits for it)
};
static_assert(sizeof(GdDecArgs<kCapLarge>) <= 18000, "kernel-argument budget");
// verdict << 48 | first offending message << 32 | its header
constexpr unsigned long long kVerdictGood = 1ull, kVerdictLong = 2ull, kVerdictShort = 3ull;

// Whether every header of the table fits its message (the same answer in all lanes of the workgroup, all of which
// must call).  `tell`: this workgroup reports.
template <int CAP>
__device__ __forceinline__ bool headers_fit(const GdDecArgs<CAP>& a, bool tell) {
  static_assert(CAP <= kThreads, "a message per lane");
  __shared__ uint32_t s_bad;
  if (threadIdx.x == 0) s_bad = 0xFFFFFFFFu;
  __syncthreads();
  const uint32_t t = threadIdx.x;
  int32_t M = 4, room = 4;
  if (t < uint32_t(a.nseg)) {
    M = *reinterpret_cast<const int32_t*>(a.seg[t].in);
    room = a.seg[t].in_size;
    if (room < M || M < 4) atomicMin(&s_bad, t);
  }
  __syncthreads();
  const uint32_t bad = s_bad;
  if (tell && a.report != nullptr && t == (bad == 0xFFFFFFFFu ? 0u : bad)) {
    const unsigned long long verdict = bad == 0xFFFFFFFFu ? kVerdictGood : room < M ? kVerdictLong : kVerdictShort;
    __hip_atomic_store(a.report, verdict << 48 | (unsigned long long)(bad & 0xFFFFu) << 32 | (unsigned long long)(uint32_t(M)),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  return bad == 0xFFFFFFFFu;
}

template <int CAP>
__global__ __launch_bounds__(kThreads) void gd_check_kernel(const GdDecArgs<CAP> a) {
  (void)headers_fit<CAP>(a, true);
}

// The fill of a written tensor is a pure write stream: streaming stores, three workgroups per CU (hpx_common.h;
// 138 M elements: 119 -> 95 us for the whole call, 103 without the limit on the workgroups), 4 KB per workgroup.
constexpr uint32_t kZeroTile = kThreads * 4;
template <int CAP>
__global__ __launch_bounds__(kThreads) void gd_zero_kernel(const GdDecArgs<CAP> a) {
  if (a.check && !headers_fit<CAP>(a, blockIdx.x == 0)) return;
  const int s = find_segment<CAP>(a.tile_start, a.nseg, blockIdx.x);
  float* __restrict__ out = a.seg[s].out;
  const uint32_t n = a.seg[s].out_n;
  const uint32_t e = uint32_t(int(blockIdx.x) - a.tile_start[s]) * kZeroTile + threadIdx.x * 4;
  if (e >= n) return;
  if (n - e >= 4) {
    st4_stream(out + e, make_float4(0.f, 0.f, 0.f, 0.f));
  } else {
    for (uint32_t i = e; i < n; i++) out[i] = 0.f;
  }
}

constexpr uint32_t kScatterBlocks = 4096;  // workgroups of one message at most; they stride over the rest
template <int CAP>
__global__ __launch_bounds__(kThreads) void gd_scatter_kernel(const GdDecArgs<CAP> a) {
  if (a.check && !headers_fit<CAP>(a, blockIdx.x == 0)) return;
  const int s = find_segment<CAP>(a.tile_start, a.nseg, blockIdx.x);
  const uint8_t* __restrict__ in = a.seg[s].in;
  float* __restrict__ out = a.seg[s].out;
  const uint32_t n = a.seg[s].out_n;
  const bool add = a.seg[s].add != 0;
  const uint32_t k = uint32_t(*reinterpret_cast<const int32_t*>(in) - 4) / 8u;
  const int32_t* __restrict__ idx = reinterpret_cast<const int32_t*>(in + 4);
  const float* __restrict__ val = reinterpret_cast<const float*>(in + 4 + size_t(k) * 4);
  const uint32_t stride = uint32_t(a.tile_start[s + 1] - a.tile_start[s]) * kThreads;
  for (uint32_t x = uint32_t(int(blockIdx.x) - a.tile_start[s]) * kThreads + threadIdx.x; x < k; x += stride) {
    const uint32_t i = uint32_t(idx[x]);
    const float v = val[x];
    if (i >= n) continue;  // not an index an encoder writes
    if (add) out[i] += v; else out[i] = v;  // gd_body.h:250, :280
  }
}

// The dynamic-LDS limit is a property of the function on one device: raised once per device (bit d of `done`:
// done on device d; devices beyond 63 set it on every call).
int allow_lds(const void* kernel, int bytes, std::atomic<uint64_t>& done) {
  int dev = 0;
  HPX_HIP(hipGetDevice(&dev));
  if (dev < 64 && (done.load(std::memory_order_acquire) >> dev & 1)) return HPX_OK;
  HPX_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
  if (dev < 64) done.fetch_or(uint64_t(1) << dev, std::memory_order_release);
  return HPX_OK;
}

// One tensor of the cut path as the host sees it.
struct CutJob {
  SortSeg seg;
  int bits;  // significant bits of its largest key (at least 1)
  int plan;  // the tensor's place among the call's plans
};

// The sort's launches for digits of BITS bits: `passes` x (count launch, scatter launch), lowest digit first, the
// last scatter writing the messages.
template <int CAP, int BITS>
int sort_passes(SortArgs<CAP>& a, int passes, hipStream_t st) {
  constexpr int kStageBytes = 2 * kSortTile * int(sizeof(uint32_t));
  static std::atomic<uint64_t> attr_done{0};
  if (const int rc = allow_lds(reinterpret_cast<const void*>(&gd_sort_pass_kernel<CAP, BITS>), kStageBytes, attr_done)) return rc;
  const dim3 grid(uint32_t(a.tile_start[a.nseg]));
  for (int pass = 0; pass < passes; pass++) {
    a.shift = pass * BITS;
    a.parity = pass & 1;
    a.last = pass == passes - 1;
    HPX_LAUNCH("gd_sort_count_kernel", (gd_sort_count_kernel<CAP, BITS>), grid, dim3(kSortThreads), st, a);
    HPX_LAUNCH_LDS("gd_sort_pass_kernel", hpx::g_prof_on, (gd_sort_pass_kernel<CAP, BITS>), grid, dim3(kSortThreads), kStageBytes, st, a);
    HPX_HIP(hipGetLastError());
  }
  return HPX_OK;
}

// The cut path of what gd_order_kernel does not take, for up to CAP tensors: the sort over all of them (as many digits as the largest key of any of
// them has; digits of 9 bits where that takes fewer passes than bytes), whose last pass writes the messages.
template <int CAP>
int sort_and_cut(const CutJob* jobs, int count, hipStream_t st) {
  SortArgs<CAP> a;
  a.nseg = count;
  int bits = 1;
  a.tile_start[0] = 0;
  for (int i = 0; i < count; i++) {
    a.seg[i] = jobs[i].seg;
    a.tile_start[i + 1] = a.tile_start[i] + int32_t(cdiv(jobs[i].seg.n, kSortTile));
    bits = jobs[i].bits > bits ? jobs[i].bits : bits;
  }
  const int bytes = (bits + 7) / 8, nines = (bits + 8) / 9;
  const int rc = nines < bytes ? sort_passes<CAP, 9>(a, nines, st) : sort_passes<CAP, 8>(a, bytes, st);
  if (rc != HPX_OK) return rc;
  return HPX_OK;
}

// The cut path in one launch.
template <int CAP>
int launch_order(const CutJob* jobs, int count, hipStream_t st) {
  SortArgs<CAP> a;
  a.nseg = count;
  a.shift = a.parity = a.last = 0;
  a.tile_start[0] = 0;
  for (int i = 0; i < count; i++) {
    a.seg[i] = jobs[i].seg;
    a.tile_start[i + 1] = a.tile_start[i] + int32_t(cdiv(jobs[i].seg.n, kWindow));
  }
  constexpr int kStageBytes = 2 * int(kCutLds) * int(sizeof(uint32_t));
  static std::atomic<uint64_t> attr_done{0};
  if (const int rc = allow_lds(reinterpret_cast<const void*>(&gd_order_kernel<CAP>), kStageBytes, attr_done)) return rc;
  HPX_LAUNCH_LDS("gd_order_kernel", hpx::g_prof_on, gd_order_kernel<CAP>, dim3(uint32_t(a.tile_start[count])), dim3(kSortThreads), kStageBytes, st, a);
  HPX_HIP(hipGetLastError());
  return HPX_OK;
}

// What the host works out per tensor before anything is launched (size arithmetic of gd_body.h:112-115, :153;
// dgc_body.h:79-80, :103).
struct Plan {
  GdSeg seg;
  size_t ws_bytes, cut_bytes;
  int margin;  // how its threshold is found: GdArgs::margin
};

// Who settles a tensor behind the pass: one workgroup (gd_finish_kernel); the expand launch and, if it has to be cut, one
// workgroup (the same launch: its LDS holds what is kept); or the expand launch and the host, which queues the cut by
// many workgroups (gd_order_kernel, or the digit sort) once it has heard the count.  The provisional path keeps to the last: it may have to fall back.
bool finishes(const GdSeg& sg, int margin) { return margin < 0 && one_workgroup(sg.n, sg.limit); }
bool cut_on_device(const GdSeg& sg, int margin) { return margin < 0 && sg.limit < kCutKeep; }

// Whether the provisional path is the quicker one for a tensor.  It saves the gather of the sample (two lines each, one
// without a residual), three of the four launches that rank it and the scan, and adds four short ones; its pass runs 8 %
// longer, the gather's lines no longer waiting for it in the cache.  us per encode and decode, gather path -> provisional, one
// in a thousand kept, by sample: 0.5 M 169.6 -> 168.2, 0.6 M 192.7 -> 184.0, 0.85 M (17 M elements) 125.8 -> 113.3, 1.38 M 377
// -> 331, 5 M 453 -> 280; 3 in a thousand: 0.6 M 149.6 -> 136.1 (30 M elements) and 209 -> 196 (60 M).  Encode without a
// residual: 0.6 M 105.2 -> 108.3, 0.8 M 125.7 -> 117.1.  Its own launches look at what is kept, and in smaller tensors longer at
// each (gd_invert_kernel): one in a hundred, 0.6 M (31 M elements) 170.0 -> 178.5, 0.9 M 24 M elements 156.6 -> 158.4 and 90 M
// 371 -> 360, 1.0 M 20 M elements 152 -> 155 and 50 M 250 -> 230, 1.5 M (76 M) 355 -> 311, 2.4 M (24 M) 223 -> 199, 5 M (100 M)
// 557 -> 479; 5 in a thousand, 1.2 M 404 -> 379 (120 M).  Beyond 12 in 1024 there are no lists (list_room).
constexpr uint32_t kProvisionalFrom = 600000, kProvisionalFromBare = 800000;   // samples ...
constexpr uint32_t kProvisionalKept = 300;                                     // ... where one element in so many is kept at most
constexpr uint32_t kProvisionalFromDense = 1000000, kProvisionalDense = 24000000;   // samples, and elements, where more are
bool provisional_pays(const GdSeg& sg, bool residual) {
  if (sg.n < kInverseFrom || sg.limit < kCutKeep || list_room(sg.n, sg.limit) == 0) return false;
  if (sg.limit <= sg.n / kProvisionalKept) return sg.sample_cnt >= (residual ? kProvisionalFrom : kProvisionalFromBare);
  return residual && sg.n >= kProvisionalDense && sg.sample_cnt >= kProvisionalFromDense;
}

// The phases for up to CAP tensors, no host wait.  margin < 0: the threshold from the full gathered sample
// (for samples of up to kPickMax one workgroup each, behind a gather launch where a sample exceeds kPickGather; for
// larger ones gather, three histogram passes, rank search), then the pass, and the finish or scan and expand.  A launch that no tensor of the table takes part in is left out.  margin >= 0: the provisional
// path (above): provisional threshold, the pass, the candidates that are samples, exact threshold, recount, expand.
template <int CAP>
int launch_phases(const Plan* plans, int count, bool residual, int margin, uint32_t* report, hipStream_t st) {
  GdArgs<CAP> a;
  a.nseg = count;
  a.residual = residual ? 1 : 0;
  a.margin = margin;
  a.gather = 0;
  a.device_cut = margin < 0 ? 1 : 0;
  a.listed = 0;
  a.report = report;
  for (int i = 0; i < count; i++) a.seg[i] = plans[i].seg;
  auto tiles = [&](auto per_tensor) {
    a.tile_start[0] = 0;
    for (int i = 0; i < count; i++) a.tile_start[i + 1] = a.tile_start[i] + int32_t(per_tensor(a.seg[i]));
    return dim3(uint32_t(a.tile_start[count]));
  };
  auto sel_blocks = [](const GdSeg& sg) {
    if (sg.sample_cnt <= kPickMax) return 0u;
    const uint32_t b = cdiv(sg.sample_cnt, kSelThreads * 8);
    return b > uint32_t(kSelBlocksMax) ? uint32_t(kSelBlocksMax) : b;
  };
  auto stream_pass = [&]() {
    const dim3 g = tiles([](const GdSeg& sg) { return cdiv(sg.n, kTile); });
    bool lists = false;
    for (int i = 0; i < count; i++) lists = lists || list_room(a.seg[i].n, a.seg[i].limit) != 0;
    auto pass = [&](auto kernel) { HPX_LAUNCH("gd_stream_kernel", kernel, g, dim3(kThreads), st, a); };
    if (margin >= 0) pass(residual ? gd_stream_kernel<true, true, true, CAP> : gd_stream_kernel<false, true, true, CAP>);
    else if (lists) pass(residual ? gd_stream_kernel<true, false, true, CAP> : gd_stream_kernel<false, false, true, CAP>);
    else pass(residual ? gd_stream_kernel<true, false, false, CAP> : gd_stream_kernel<false, false, false, CAP>);
  };
  constexpr int kStageBytes = 2 * int(kCutLds) * int(sizeof(uint32_t));   // of the finish
  dim3 grid;
  if (margin < 0) {
    // One workgroup's gathers of a sample take as long as a launch that spreads them at about kPickGather samples;
    // beside larger samples that launch is there anyway.
    a.gather = kPickGather;
    for (int i = 0; i < count; i++)
      if (a.seg[i].sample_cnt > kPickGather) a.gather = kPickGatherBeside;
    const uint32_t gather = a.gather;
    grid = tiles([gather](const GdSeg& sg) {
      if (sg.sample_cnt <= gather) return 0u;
      return cdiv(sg.sample_cnt, kThreads);   // more than enough lanes to clear the histograms where they are used
    });
    if (grid.x) HPX_LAUNCH("gd_sample_kernel", gd_sample_kernel<CAP>, grid, dim3(kThreads), st, a);
    grid = tiles([](const GdSeg& sg) { return sg.sample_cnt <= kPickMax ? 1u : 0u; });
    if (grid.x) HPX_LAUNCH("gd_pick_kernel", gd_pick_kernel<CAP>, grid, dim3(kSelThreads), st, a);
    grid = tiles(sel_blocks);
    if (grid.x) {
      HPX_LAUNCH("gd_select_kernel", (gd_select_kernel<1, CAP>), grid, dim3(kSelThreads), st, a);
      HPX_LAUNCH("gd_select_kernel", (gd_select_kernel<2, CAP>), grid, dim3(kSelThreads), st, a);
      HPX_LAUNCH("gd_select_kernel", (gd_select_kernel<3, CAP>), grid, dim3(kSelThreads), st, a);
      grid = tiles([](const GdSeg& sg) { return sg.sample_cnt <= kPickMax ? 0u : 1u; });
      HPX_LAUNCH("gd_threshold_kernel", gd_threshold_kernel<CAP>, grid, dim3(kSelThreads), st, a);
    }
    // Before the pass, which leaves zeros in the residual for what the finish sends (clears_listed); behind the first launches, which it need not hold up.
    static std::atomic<uint64_t> attr_done{0};
    if (const int rc = allow_lds(reinterpret_cast<const void*>(&gd_finish_kernel<CAP>), kStageBytes, attr_done)) return rc;
    stream_pass();
  } else {
    grid = tiles([](const GdSeg& sg) { return cdiv(pre_samples(sg.sample_cnt, sg.thr_index), kThreads); });
    HPX_LAUNCH("gd_presample_kernel", gd_presample_kernel<CAP>, grid, dim3(kThreads), st, a);
    HPX_LAUNCH("gd_prepick_kernel", gd_prepick_kernel<CAP>, dim3(uint32_t(count)), dim3(kThreads), st, a);
    stream_pass();
    grid = tiles([](const GdSeg& sg) { return sg.n < kInverseFrom ? cdiv(sg.sample_cnt, kThreads) : cdiv(cdiv(sg.n, kTile), kExpandPerBlock); });
    HPX_LAUNCH("gd_invert_kernel", gd_invert_kernel<CAP>, grid, dim3(kThreads), st, a);
    HPX_LAUNCH("gd_exact_kernel", gd_exact_kernel<CAP>, dim3(uint32_t(count)), dim3(kSelThreads), st, a);
    grid = tiles([](const GdSeg& sg) { return cdiv(cdiv(sg.n, kTile), kExpandPerBlock); });
    HPX_LAUNCH("gd_recount_kernel", gd_recount_kernel<CAP>, grid, dim3(kThreads), st, a);
  }
  grid = tiles([margin](const GdSeg& sg) {
    const uint32_t chunks = cdiv(cdiv(sg.n, kTile), kScanChunk);
    return margin < 0 && chunks > 1 ? chunks : 0u;
  });
  if (grid.x) HPX_LAUNCH("gd_scan_kernel", gd_scan_kernel<CAP>, grid, dim3(kSelThreads), st, a);
  HPX_HIP(hipGetLastError());
  // Queued before the host knows the counts: the finish where nothing has to be cut,
  // else the candidate list and keys of the cut path.
  grid = tiles([margin](const GdSeg& sg) { return finishes(sg, margin) ? 0u : cdiv(cdiv(sg.n, kTile), kExpandPerBlock); });
  if (grid.x) HPX_LAUNCH("gd_expand_kernel", gd_expand_kernel<CAP>, grid, dim3(kThreads), st, a);
  grid = tiles([margin](const GdSeg& sg) { return finishes(sg, margin) || cut_on_device(sg, margin) ? 1u : 0u; });
  if (grid.x) {
    HPX_LAUNCH_LDS("gd_finish_kernel", hpx::g_prof_on, gd_finish_kernel<CAP>, grid, dim3(kSortThreads), kStageBytes, st, a);
  }
  HPX_HIP(hipGetLastError());
  return HPX_OK;
}

// Polls pinned host memory until `pending` is false.  Every 2 ms it also asks whether the stream has drained, which ends the
// wait if the words can only be seen once the kernels have finished, or if a launch failed.  Not more often: asking puts
// work of its own on the stream (asked every 512 polls, about 7 us, a call on one tensor of a million took 40.4 us, now 32.8).
// HPX_OK also where everything has run and nothing came: the caller looks.
constexpr std::chrono::milliseconds kAskEvery(2);
template <typename Pending>
int poll_memory(Pending pending, const char* who, hipStream_t st) {
  auto asked = std::chrono::steady_clock::now();
  for (uint32_t spins = 1; pending(); spins++) {
    _mm_pause();
    if ((spins & 511u) != 0) continue;
    const auto now = std::chrono::steady_clock::now();
    if (now - asked < kAskEvery) continue;
    asked = now;
    const hipError_t e = hipStreamQuery(st);
    if (e == hipErrorNotReady) { (void)hipGetLastError(); continue; }
    if (e != hipSuccess) {
      hpx::set_error("%s: the stream failed: %s", who, hipGetErrorString(e));
      return HPX_ERR_HIP;
    }
    break;
  }
  __atomic_thread_fence(__ATOMIC_ACQUIRE);
  return HPX_OK;
}

// Waits until the expand launch has reported every tensor of `count` (the words are in pinned host memory and
// the kernel writes them with system-scope stores as the first thing it does, so they arrive while the stream
// is still busy with that launch).  A tensor that is settled on the device is not waited for.
int wait_reports(volatile uint32_t* report, const Plan* plans, int count, hipStream_t st) {
  for (int t = 0; t < count; t++) {
    if (cut_on_device(plans[t].seg, plans[t].margin)) continue;
    volatile uint32_t* word = report + size_t(t) * kReportWords;
    auto pending = [word]() { return word[0] == kNotReported || word[1] == kNotReported || word[2] == kNotReported; };
    const int rc = poll_memory(pending, "sparsifier encode", st);
    if (rc != HPX_OK) return rc;
    if (pending()) {  // everything has run and still no report
      hpx::set_error("sparsifier encode: tensor %d was not reported by the expand launch", t);
      return HPX_ERR_HIP;
    }
  }
  return HPX_OK;
}

// The same for one 64-bit word that is zero until a kernel writes it.
int wait_word(volatile unsigned long long* word, hipStream_t st) {
  const int rc = poll_memory([word]() { return *word == 0; }, "sparsifier decode", st);
  if (rc != HPX_OK) return rc;
  if (*word == 0) {
    hpx::set_error("sparsifier decode: the headers were not reported");
    return HPX_ERR_HIP;
  }
  return HPX_OK;
}

// Whether the windows are quicker than the digit sort for what a call has to cut, all of it one way or the other.  The sort shares
// its launches among the tensors; the windows queue up, one for each CU at a time, and each reads all the keys of its tensor.  us per
// encode of tensors with zeros around their candidates, sort / windows (keys read in all by the windows; their number):
//   4 tensors of 130 thousand candidates 117 / 105 (66 M; 508), 5 of 120 thousand 124 / 122 (71 M; 590), 12 of 90 thousand 173 / 173 (95 M; 1056),
//   2 of 220 thousand 118 / 119 (95 M; 430), 4 of 160 thousand 123 / 130 (101 M), 5 of 150 thousand 133 / 144 (110 M),
//   10 of 220 thousand 221 / 312;
//   100 of 9 thousand 168 / 147 (900), 50 of 30 thousand 204 / 190 (1500), 200 of 9 thousand 245 / 240 (1800), 100 of 20 thousand 243 / 256 (2000),
//   200 of 12 thousand 299 / 311 (2400).
// Where one tensor has to be sorted, or has hardly any candidates, the others go with it: one of 240 thousand and five of 50 thousand 124, with these
// in windows 138; one of 300 thousand and five of 10 thousand 124 and 147.
constexpr uint64_t kOrderKeys = 90u << 20;        // read by the windows of a call ...
constexpr uint32_t kOrderWindows = 7 * 256;       // ... and how many of them
bool windows_pay(const std::vector<CutJob>& jobs) {
  uint64_t keys = 0, windows = 0;
  for (const CutJob& job : jobs) {
    if (job.seg.n < kWindowSample || job.seg.n > kOrderMax) return false;
    const uint64_t w = cdiv(job.seg.n, kWindow);
    windows += w;
    keys += w * job.seg.n;
  }
  return keys <= kOrderKeys && windows <= kOrderWindows;
}

constexpr int kMaxPerWait = int((hpx::kPinnedFlagOffset) / (kReportWords * sizeof(uint32_t)));  // tensors whose reports fit the pinned block

// `count` tensors.  With residuals (`residuals` non-null): gd_body, s_percent = 1 - drop_ratio.  Without:
// dgc_with_auxiliary_body, where the gradient itself is thresholded and its selected entries cleared.
// A tensor whose parameters make no sense is reported and skipped, like the reference driver's
// print-and-continue; the others are encoded.
int gd_encode_batch(int count, float* const* grads, const int32_t* Ns, float* const* residuals, uint8_t* const* outs,
                    const double* sample_rates, const double* s_percents, const uint64_t* seeds, hpx::Workspace* ws,
                    hipStream_t st) {
  int worst = HPX_OK;
  std::vector<Plan> plans;
  plans.reserve(count);
  size_t ws_total = 0;
  for (int i = 0; i < count; i++) {
    const int32_t N = Ns[i];
    const int32_t sample_cnt = static_cast<int32_t>(std::ceil(N * sample_rates[i]));
    const int32_t expected = static_cast<int32_t>(std::ceil(N * s_percents[i]));
    const int32_t thr_index = static_cast<int32_t>(sample_cnt * s_percents[i]);
    if (!(sample_cnt > 0 && thr_index >= 0 && thr_index < sample_cnt && expected >= 0)) {
      hpx::set_error("sparsifier encode: tensor %d: N=%d sample_rate=%g kept fraction=%g give sample_cnt=%d threshold index=%d", i,
                     N, sample_rates[i], s_percents[i], sample_cnt, thr_index);
      if (worst == HPX_OK) worst = HPX_ERR_ARG;
      continue;
    }
    Plan p;
    const uint32_t n = static_cast<uint32_t>(N);
    // Room for the cut path is laid out for a typical overshoot before anything is
    // launched: the expand kernel fills it without the host knowing the count.
    uint64_t cap64 = uint64_t(expected) * 2 > uint64_t(expected) + 65536 ? uint64_t(expected) * 2 : uint64_t(expected) + 65536;
    if (cap64 > n) cap64 = n;
    const uint64_t seed = seeds ? seeds[i] : hpx::clock_seed();
    p.seg.g = grads[i];
    p.seg.r = residuals ? residuals[i] : grads[i];
    p.seg.out = outs[i];
    p.seg.ws = nullptr;
    p.seg.cut = nullptr;
    p.seg.n = n;
    p.seg.sample_cnt = static_cast<uint32_t>(sample_cnt);
    p.seg.seed = static_cast<uint32_t>(seed);
    p.seg.thr_index = static_cast<uint32_t>(thr_index);
    p.seg.limit = static_cast<uint32_t>(expected);
    p.seg.cap = static_cast<uint32_t>(cap64);
    p.ws_bytes = gd_layout(n, p.seg.sample_cnt).end + list_bytes(n, p.seg.limit);
    p.cut_bytes = cut_layout(cap64).end;
    ws_total += p.ws_bytes + p.cut_bytes;
    plans.push_back(p);
  }
  if (plans.empty()) return worst;
  int rc = hpx::ensure_workspace(ws, ws_total);
  if (rc != HPX_OK) return rc;
  {
    size_t at = 0;
    for (Plan& p : plans) {
      p.seg.ws = ws->dev + at;  at += p.ws_bytes;
      p.seg.cut = ws->dev + at; at += p.cut_bytes;
    }
  }
  volatile uint32_t* report = reinterpret_cast<volatile uint32_t*>(ws->pinned);
  const int total = int(plans.size());
  uint64_t all_samples = 0;
  for (const Plan& p : plans) all_samples += p.seg.sample_cnt;
  const int64_t prov_min = hpx::option(hpx::kOptGdProvisionalMinSamples);
  const int64_t prov_margin = hpx::option(hpx::kOptGdProvisionalMargin);
  const int margin = (prov_min >= 0 && all_samples >= uint64_t(prov_min) && prov_margin >= 0) ? int(prov_margin > 1000 ? 1000 : prov_margin) : -1;
  for (Plan& p : plans) p.margin = prov_min == kProvisionalAuto ? (provisional_pays(p.seg, residuals != nullptr) ? kBySpread : -1) : margin;
  // a launch table takes tensors of one path
  std::stable_partition(plans.begin(), plans.end(), [](const Plan& p) { return p.margin >= 0; });
  auto reset_reports = [&](int n_) {
    for (int t = 0; t < n_; t++)
      for (int w = 0; w < 3; w++) report[size_t(t) * kReportWords + w] = kNotReported;
    __atomic_thread_fence(__ATOMIC_RELEASE);
  };
  for (int first = 0; first < total; first += kMaxPerWait) {
    const int batch = total - first < kMaxPerWait ? total - first : kMaxPerWait;
    reset_reports(batch);
    for (int k = 0, m; k < batch; k += m) {
      const int how = plans[first + k].margin;
      for (m = 1; m < kCapLarge && k + m < batch && plans[first + k + m].margin == how;) m++;
      uint32_t* rep = const_cast<uint32_t*>(report) + size_t(k) * kReportWords;
      rc = m <= kCapSmall ? launch_phases<kCapSmall>(&plans[first + k], m, residuals != nullptr, how, rep, st)
                          : launch_phases<kCapLarge>(&plans[first + k], m, residuals != nullptr, how, rep, st);
      if (rc != HPX_OK) return rc;
    }
    rc = wait_reports(report, &plans[first], batch, st);
    if (rc != HPX_OK) return rc;
    // What the tensors reported, kept on the host: the pinned words serve again below.
    std::vector<uint32_t> rep_host(size_t(batch) * kReportWords);
    for (size_t w = 0; w < rep_host.size(); w++) rep_host[w] = report[w];
    if (plans[first].margin >= 0) {   // those come first
      // Tensors whose provisional threshold lies above the exact one: through the gather path, on the array
      // the pass has already updated (it holds G + R now: sampled and thresholded as it is, nothing added again).
      std::vector<int> fb;
      for (int t = 0; t < batch; t++)
        if (rep_host[size_t(t) * kReportWords] == kFallback) fb.push_back(t);
      if (!fb.empty()) {
        std::vector<Plan> again;
        for (int t : fb) {
          Plan p = plans[first + t];
          p.seg.g = p.seg.r;
          p.margin = plans[first + t].margin = -1;
          again.push_back(p);
        }
        ws->gd_fallbacks += fb.size();
        reset_reports(int(again.size()));
        for (size_t k = 0; k < again.size(); k += kCapLarge) {
          const int m = int(again.size() - k < size_t(kCapLarge) ? again.size() - k : size_t(kCapLarge));
          uint32_t* rep = const_cast<uint32_t*>(report) + k * kReportWords;
          rc = m <= kCapSmall ? launch_phases<kCapSmall>(&again[k], m, false, -1, rep, st)
                              : launch_phases<kCapLarge>(&again[k], m, false, -1, rep, st);
          if (rc != HPX_OK) return rc;
        }
        rc = wait_reports(report, again.data(), int(again.size()), st);
        if (rc != HPX_OK) return rc;
        for (size_t j = 0; j < fb.size(); j++) {
          for (int w = 0; w < kReportWords; w++) rep_host[size_t(fb[j]) * kReportWords + w] = report[j * kReportWords + w];
          if (cut_on_device(again[j].seg, -1)) rep_host[size_t(fb[j]) * kReportWords] = 0;   // nothing left to cut
        }
      }
    }
    // More candidates than `expected`: order them by |r| descending and keep the first `expected`
    // (gd_body.h:176-187), all such tensors of the batch together.
    std::vector<CutJob> jobs;
    std::vector<int> overflow;   // jobs whose candidates are more than their buffers were laid out for
    size_t aux_need = 0;
    for (int t = 0; t < batch; t++) {
      const GdSeg& sg = plans[first + t].seg;
      const uint32_t found = rep_host[size_t(t) * kReportWords];
      if (cut_on_device(sg, plans[first + t].margin) || found <= sg.limit) continue;
      const uint32_t thr_bits = rep_host[size_t(t) * kReportWords + 1], max_bits = rep_host[size_t(t) * kReportWords + 2];
      // keys are |r| bits minus threshold bits: the largest tells how many byte digits are in use
      const uint32_t max_key = max_bits > thr_bits ? max_bits - thr_bits : 0u;
      CutJob job;
      job.bits = max_key ? 32 - __builtin_clz(max_key) : 1;
      job.seg.msg = sg.out;
      job.seg.r = sg.r;
      job.seg.n = found;
      job.seg.keep = sg.limit;
      job.seg.thr_bits = thr_bits;
      job.seg.cut = sg.cut;
      job.seg.cap = sg.cap;
      job.plan = first + t;
      if (found > sg.cap) {
        overflow.push_back(int(jobs.size()));
        aux_need += cut_layout(found).end;
      }
      jobs.push_back(job);
    }
    if (!overflow.empty()) {
      // Far more candidates than reserved for: list them again into a block of their own.
      rc = hpx::ensure_aux(ws, aux_need);
      if (rc != HPX_OK) return rc;
      size_t at = 0;
      for (int j : overflow) {
        CutJob& job = jobs[j];
        const Plan& plan = plans[job.plan];
        job.seg.cut = ws->aux + at;
        job.seg.cap = job.seg.n;
        at += cut_layout(job.seg.n).end;
        GdArgs<kCapSmall> a;
        a.nseg = 1;
        a.residual = residuals != nullptr;
        a.margin = plan.margin;   // where its offsets come from
        a.gather = 0;
        a.device_cut = 0;
        a.listed = plan.seg.limit;
        a.report = nullptr;  // the host has its report
        a.seg[0] = plan.seg;
        a.seg[0].cut = job.seg.cut;
        a.seg[0].cap = job.seg.n;
        a.seg[0].limit = 0u;
        a.tile_start[0] = 0;
        a.tile_start[1] = int32_t(cdiv(cdiv(plan.seg.n, kTile), kExpandPerBlock));
        HPX_LAUNCH("gd_expand_kernel", gd_expand_kernel<kCapSmall>, dim3(uint32_t(a.tile_start[1])), dim3(kThreads), st, a);
        HPX_HIP(hipGetLastError());
      }
    }
    const bool windows = windows_pay(jobs);
    for (size_t k = 0; k < jobs.size(); k += kCapLarge) {
      const int m = int(jobs.size() - k < size_t(kCapLarge) ? jobs.size() - k : size_t(kCapLarge));
      if (windows) rc = m <= kCapSmall ? launch_order<kCapSmall>(&jobs[k], m, st) : launch_order<kCapLarge>(&jobs[k], m, st);
      else rc = m <= kCapSmall ? sort_and_cut<kCapSmall>(&jobs[k], m, st) : sort_and_cut<kCapLarge>(&jobs[k], m, st);
      if (rc != HPX_OK) return rc;
    }
  }
  return worst;
}

}  // namespace

HPX_API int hpx_gd_encode(int count, const float* const* grads, const int32_t* Ns, float* const* residuals,
                          uint8_t* const* outs, const double* sample_rates, const double* drop_ratios,
                          const uint64_t* seeds, hpx_stream_t stream) {
  hpx::clear_error();
  HPX_ARG(count >= 0, "hpx_gd_encode: negative count");
  if (count == 0) return HPX_OK;
  HPX_ARG(grads && Ns && residuals && outs && sample_rates && drop_ratios, "hpx_gd_encode: null argument array");
  for (int i = 0; i < count; i++) {
    HPX_ARG(Ns[i] > 0, "hpx_gd_encode: tensor %d has size %d (must be positive)", i, Ns[i]);
    HPX_ARG(grads[i] && residuals[i] && outs[i], "hpx_gd_encode: tensor %d has a null pointer", i);
    HPX_ARG((reinterpret_cast<uintptr_t>(outs[i]) & 3) == 0, "hpx_gd_encode: output %d is not 4-byte aligned", i);
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (const int rcc = hpx::reject_capture(st, "hpx_gd_encode")) return rcc;
  hpx::Workspace* ws = hpx::workspace_record(st);
  if (!ws) return HPX_ERR_HIP;
  std::lock_guard<std::mutex> lock(ws->mu);
  std::vector<double> kept(count);
  for (int i = 0; i < count; i++) kept[i] = 1 - drop_ratios[i];  // s_percent, gd_body.h:112
  return gd_encode_batch(count, const_cast<float* const*>(grads), Ns, residuals, outs, sample_rates, kept.data(), seeds, ws, st);
}

HPX_API int64_t hpx_gd_fallbacks(hpx_stream_t stream) {
  hpx::clear_error();
  hpx::Workspace* ws = hpx::workspace_record(static_cast<hipStream_t>(stream));
  if (!ws) return -1;
  std::lock_guard<std::mutex> lock(ws->mu);
  return int64_t(ws->gd_fallbacks);
}

namespace {
// A table of messages, none of which names another's output.
template <int CAP>
void decode_table(GdDecArgs<CAP>& a, const GdMsg* msgs, int count, bool check, unsigned long long* report) {
  a.nseg = count;
  a.check = check ? 1 : 0;
  a.report = report;
  for (int i = 0; i < count; i++) a.seg[i] = msgs[i];
}
template <int CAP>
int launch_check(const GdMsg* msgs, int count, unsigned long long* report, hipStream_t st) {
  GdDecArgs<CAP> a;
  decode_table(a, msgs, count, true, report);
  a.tile_start[0] = 0;
  for (int i = 0; i < count; i++) a.tile_start[i + 1] = 0;
  HPX_LAUNCH("gd_check_kernel", gd_check_kernel<CAP>, dim3(1), dim3(kThreads), st, a);
  HPX_HIP(hipGetLastError());
  return HPX_OK;
}
// The fill of the tensors that are written (zero_fill), then all values to their places.
template <int CAP>
int launch_decode(const GdMsg* msgs, int count, bool zero_fill, bool check, unsigned long long* report, hipStream_t st) {
  GdDecArgs<CAP> a;
  decode_table(a, msgs, count, check, report);
  a.tile_start[0] = 0;
  for (int i = 0; i < count; i++)
    a.tile_start[i + 1] = a.tile_start[i] + (zero_fill && !msgs[i].add ? int32_t(cdiv(msgs[i].out_n, kZeroTile)) : 0);
  if (a.tile_start[count] > 0) {
    HPX_LAUNCH_LDS("gd_zero_kernel", hpx::g_prof_on, gd_zero_kernel<CAP>, dim3(uint32_t(a.tile_start[count])), dim3(kThreads),
                   hpx::kWriteStreamPadLds3, st, a);
    a.report = nullptr;  // that launch reports
  }
  for (int i = 0; i < count; i++) {
    // by the room the message has: its header is on the device
    const uint32_t most = cdiv(msgs[i].in_size > 4 ? uint32_t(msgs[i].in_size - 4) / 8u : 0u, kThreads);
    a.tile_start[i + 1] = a.tile_start[i] + int32_t(most < 1 ? 1 : most > kScatterBlocks ? kScatterBlocks : most);
  }
  HPX_LAUNCH("gd_scatter_kernel", gd_scatter_kernel<CAP>, dim3(uint32_t(a.tile_start[count])), dim3(kThreads), st, a);
  HPX_HIP(hipGetLastError());
  return HPX_OK;
}

// gd_r_body (zero_fill: write mode clears the whole output first, gd_body.h:335-347)
// and dgc_r_body (no clearing, dgc_body.h:283-289).
int decode_messages(int count, const uint8_t* const* ins, const int32_t* in_sizes, float* const* outs,
                    const int32_t* out_sizes, const int32_t* is_add_tos, bool zero_fill, hpx_stream_t stream) {
  hpx::clear_error();
  HPX_ARG(count >= 0, "hpx_gd_decode: negative count");
  if (count == 0) return HPX_OK;
  HPX_ARG(ins && in_sizes && outs && out_sizes && is_add_tos, "hpx_gd_decode: null argument array");
  // the headers are read back into the pinned block, whose last words belong to the barrier kernels' expiry flag
  HPX_ARG(size_t(count) * sizeof(int32_t) <= hpx::kPinnedFlagOffset, "hpx_gd_decode: more than %zu messages in one call",
          hpx::kPinnedFlagOffset / sizeof(int32_t));
  for (int i = 0; i < count; i++) {
    HPX_ARG(ins[i] && outs[i] && out_sizes[i] >= 0, "hpx_gd_decode: message %d has a null pointer or negative size", i);
    HPX_ARG((reinterpret_cast<uintptr_t>(ins[i]) & 3) == 0, "hpx_gd_decode: message %d is not 4-byte aligned", i);
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (const int rcc = hpx::reject_capture(st, zero_fill ? "hpx_gd_decode" : "hpx_dgc_decode")) return rcc;
  hpx::Workspace* ws = hpx::workspace_record(st);
  if (!ws) return HPX_ERR_HIP;
  std::lock_guard<std::mutex> lock(ws->mu);
  int rc = hpx::ensure_workspace(ws, 0);
  if (rc != HPX_OK) return rc;

  // Messages that name one output are applied in call order: round j takes the j-th message of every output, all of a
  // round together; outputs that overlap otherwise take a round per message.
  std::vector<int> order(count), round_of(count, 0);
  for (int i = 0; i < count; i++) order[i] = i;
  int rounds = 1;
  if (const int cls = hpx::classify_outputs(count, outs, out_sizes)) {
    std::unordered_map<const float*, int> seen;
    for (int i = 0; i < count; i++) {
      round_of[i] = cls == 1 ? seen[outs[i]]++ : i;
      rounds = round_of[i] + 1 > rounds ? round_of[i] + 1 : rounds;
    }
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return round_of[x] < round_of[y]; });
  }
  uint64_t zero_tiles = 0;
  for (int i = 0; i < count; i++)
    if (zero_fill && !is_add_tos[i]) zero_tiles += cdiv(uint32_t(out_sizes[i]), kZeroTile);

  std::vector<GdMsg> msgs(count);
  for (int i = 0; i < count; i++) msgs[i] = {ins[i], outs[i], static_cast<uint32_t>(out_sizes[i]), in_sizes[i], is_add_tos[i], 0};

  volatile unsigned long long* report = reinterpret_cast<volatile unsigned long long*>(ws->pinned);
  // One table and hardly anything to clear: everything is queued at once and checks for itself.  Else the host
  // hears the verdict first (about 6 us): a fill of many short workgroups is slowed by reading headers in each
  // (from about a thousand workgroups on, more than the wait costs), and several tables must all be good before any is applied.
  const bool at_once = rounds == 1 && count <= kCapLarge && zero_tiles <= 1024;
  const int tables = at_once ? 1 : (count + kCapLarge - 1) / kCapLarge;
  for (int k = 0; k < tables; k++) report[k] = 0;
  __atomic_thread_fence(__ATOMIC_RELEASE);
  auto verdict = [&]() {
    for (int k = 0; k < tables; k++) {
      const int rcw = wait_word(&report[k], st);
      if (rcw != HPX_OK) return rcw;
      const unsigned long long w = report[k];
      if ((w >> 48) == kVerdictGood) continue;
      const int i = k * kCapLarge + int(w >> 32 & 0xFFFFu);
      const int32_t M = static_cast<int32_t>(uint32_t(w));
      if ((w >> 48) == kVerdictLong) {  // gd_body.h:317-325
        hpx::set_error("input space provided is not enough! in_uint8_t_size=%d\tM=%d (message %d, is_add_to %d)", in_sizes[i], M, i,
                       is_add_tos[i]);
        return int(HPX_ERR_BODY);
      }
      hpx::set_error("hpx_gd_decode: message %d has header %d", i, M);
      return int(HPX_ERR_ARG);
    }
    return int(HPX_OK);
  };
  unsigned long long* word = reinterpret_cast<unsigned long long*>(ws->pinned);
  if (at_once) {
    rc = count <= kCapSmall ? launch_decode<kCapSmall>(msgs.data(), count, zero_fill, true, word, st)
                            : launch_decode<kCapLarge>(msgs.data(), count, zero_fill, true, word, st);
    return rc != HPX_OK ? rc : verdict();
  }
  for (int k = 0; k < count; k += kCapLarge) {
    const int m = count - k < kCapLarge ? count - k : kCapLarge;
    rc = m <= kCapSmall ? launch_check<kCapSmall>(&msgs[k], m, word + k / kCapLarge, st)
                        : launch_check<kCapLarge>(&msgs[k], m, word + k / kCapLarge, st);
    if (rc != HPX_OK) return rc;
  }
  rc = verdict();
  if (rc != HPX_OK) return rc;
  std::vector<GdMsg> sorted(count);
  for (int i = 0; i < count; i++) sorted[i] = msgs[order[i]];
  for (int first = 0; first < count;) {
    // a round at most, and no more workgroups than a launch takes
    int last = first;
    uint64_t tiles = 0;
    while (last < count && last - first < kCapLarge && round_of[order[last]] == round_of[order[first]]) {
      tiles += cdiv(sorted[last].out_n, kZeroTile) + kScatterBlocks;
      if (last > first && tiles > (1u << 23)) break;
      last++;
    }
    rc = last - first <= kCapSmall ? launch_decode<kCapSmall>(&sorted[first], last - first, zero_fill, false, nullptr, st)
                                   : launch_decode<kCapLarge>(&sorted[first], last - first, zero_fill, false, nullptr, st);
    if (rc != HPX_OK) return rc;
    first = last;
  }
  return HPX_OK;
}
}  // namespace

HPX_API int hpx_gd_decode(int count, const uint8_t* const* ins, const int32_t* in_sizes, float* const* outs,
                          const int32_t* out_sizes, const int32_t* is_add_tos, hpx_stream_t stream) {
  return decode_messages(count, ins, in_sizes, outs, out_sizes, is_add_tos, true, stream);
}

HPX_API int hpx_dgc_decode(int count, const uint8_t* const* ins, const int32_t* in_sizes, float* const* outs,
                           const int32_t* out_sizes, const int32_t* is_add_tos, hpx_stream_t stream) {
  return decode_messages(count, ins, in_sizes, outs, out_sizes, is_add_tos, false, stream);
}

HPX_API int hpx_dgc_encode(int count, float* const* grads, const int32_t* Ns, uint8_t* const* outs,
                           const double* sample_rates, const double* s_percents, const uint64_t* seeds,
                           hpx_stream_t stream) {
  hpx::clear_error();
  HPX_ARG(count >= 0, "hpx_dgc_encode: negative count");
  if (count == 0) return HPX_OK;
  HPX_ARG(grads && Ns && outs && sample_rates && s_percents, "hpx_dgc_encode: null argument array");
  for (int i = 0; i < count; i++) {
    HPX_ARG(Ns[i] > 0, "hpx_dgc_encode: tensor %d has size %d (must be positive)", i, Ns[i]);
    HPX_ARG(grads[i] && outs[i], "hpx_dgc_encode: tensor %d has a null pointer", i);
    HPX_ARG((reinterpret_cast<uintptr_t>(outs[i]) & 3) == 0, "hpx_dgc_encode: output %d is not 4-byte aligned", i);
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (const int rcc = hpx::reject_capture(st, "hpx_dgc_encode")) return rcc;
  hpx::Workspace* ws = hpx::workspace_record(st);
  if (!ws) return HPX_ERR_HIP;
  std::lock_guard<std::mutex> lock(ws->mu);
  return gd_encode_batch(count, grads, Ns, nullptr, outs, sample_rates, s_percents, seeds, ws, st);
}
