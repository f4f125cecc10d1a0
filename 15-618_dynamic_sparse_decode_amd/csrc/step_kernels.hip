// step_kernels.hip -- the kernels of one sparse decode step (gfx950):
//   1. exact-order page scoring   (reference ScorePagesCpu, src/reference_kernels.cpp:59-80)
//   2. per-request top-k select   (reference SelectTopKPagesCpu, :82-107)
//   3. fused gather + attention: attention.hip
// and the wide step, all three in one launch.
#include <algorithm>
#include <cmath>

#include "attention_head.h"
#include "dsd_internal.h"
#include "score_slice.h"
#include "step_common.h"

namespace dsdk {
namespace {

// ---------------------------------------------------------------------------
// 1. Exact-order scoring.
//
// The reference scores a page as acc = 0; acc = fl(acc + fl(q[i]*s[i])) for
// i = 0..E-1, then fl(acc*scale).  That chain must be reproduced in order to
// keep page selection bit-exact, so one lane owns one candidate page and adds
// its products in order with separately rounded multiply and add (__fmul_rn /
// __fadd_rn; never contracted to FMA).
//
// ScoreChainsKernel (E a multiple of 64): a workgroup takes 8, 16 or 32 pages
// of one request; the lanes of its first wave run their chains from products
// that the other waves form in LDS, a stretch ahead, from rows read whole
// (RescoreChains).  Bound by the chain, E dependent adds fed from LDS at
// about 7 cycles each (E = 4096: 12 us), so a small batch takes few pages per
// workgroup and spreads them over the chip.  16 requests of 512-2048 tokens
// (1207 pages): 25 us; 108 us with the kernel below, whose 32 waves were all
// there was and read 64 rows a line at a time.
//
// ScoreExactKernel (other E, and batches of more pages than the chains kernel
// takes in one round): a wave of 64 candidates, each lane walking its own row in
// memory.
// ---------------------------------------------------------------------------
constexpr int kChainPages = 32;
constexpr int kChainThreads = 512;

__global__ __launch_bounds__(kChainThreads) void ScoreChainsKernel(
    const float* __restrict__ queries, const float* __restrict__ summaries,
    const int* __restrict__ token_counts, int capacity, const int* __restrict__ cand_offsets,
    const int* __restrict__ cand_ids, int total, int pages_per_group, int E, float scale,
    float* __restrict__ scores, const int* __restrict__ only, FailReport fail) {
  __shared__ __align__(16) float tile[RescoreFloats<kChainPages>()];
  __shared__ int s_page[kChainPages];
  const int r = blockIdx.y;
  if (only != nullptr && only[r] >= 0) return;  // decided without exact scores
  int begin, n;
  if (!RequestRange(cand_offsets, r, total, fail, &begin, &n)) return;
  const int first = static_cast<int>(blockIdx.x) * pages_per_group;
  if (first >= n) return;
  const int pages = n - first < pages_per_group ? n - first : pages_per_group;
  if (static_cast<int>(threadIdx.x) < pages) {
    // A page holding no tokens reads as an all-zero summary
    // (src/paged_kv_cache.cpp:457-459); the products q*0 are still formed.  An
    // id outside the pool scores as such a page and is reported.
    const int page = cand_ids[begin + first + threadIdx.x];
    if (!InPool(page, capacity)) ReportFailure(fail, kFailPageId);
    s_page[threadIdx.x] = page;
  }
  __syncthreads();
  RescoreChains<kChainPages, kChainThreads>(
      pages, [&](int f) { return s_page[f]; },
      [&](int f, float score) { scores[begin + first + f] = score; },
      queries + static_cast<size_t>(r) * E, summaries, token_counts, capacity, E, scale, tile);
}

template <bool kVec4>
__global__ __launch_bounds__(kWave) void ScoreExactKernel(
    const float* __restrict__ queries, const float* __restrict__ summaries,
    const int* __restrict__ token_counts, int capacity, const int* __restrict__ cand_offsets,
    const int* __restrict__ cand_ids, int total, int E, float scale,
    float* __restrict__ scores, FailReport fail) {
  const int r = blockIdx.y;
  int begin, n;
  if (!RequestRange(cand_offsets, r, total, fail, &begin, &n)) return;
  const int end = begin + n;
  const int first = begin + blockIdx.x * kWave;
  if (first >= end) return;
  const int c = first + static_cast<int>(threadIdx.x);
  const bool active = c < end;
  int page = active ? cand_ids[c] : cand_ids[first];
  // A page holding no tokens reads as an all-zero summary
  // (src/paged_kv_cache.cpp:457-459); the products q*0 are still formed.  An
  // id outside the pool scores as such a page and is reported.
  bool zero = !active;
  if (!InPool(page, capacity)) {
    if (active) ReportFailure(fail, kFailPageId);
    page = 0;
    zero = true;
  }
  zero = zero || token_counts[page] == 0;
  const float* __restrict__ q = queries + static_cast<size_t>(r) * E;
  const float* __restrict__ s = summaries + static_cast<size_t>(page) * E;

  float acc = 0.0f;
  if constexpr (kVec4) {
#pragma unroll 8
    for (int i = 0; i < E; i += 4) {
      const float4 qv = *reinterpret_cast<const float4*>(q + i);
      float4 sv = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (!zero) sv = *reinterpret_cast<const float4*>(s + i);
      acc = __fadd_rn(acc, __fmul_rn(qv.x, sv.x));
      acc = __fadd_rn(acc, __fmul_rn(qv.y, sv.y));
      acc = __fadd_rn(acc, __fmul_rn(qv.z, sv.z));
      acc = __fadd_rn(acc, __fmul_rn(qv.w, sv.w));
    }
  } else {
    for (int i = 0; i < E; ++i) {
      const float sv = zero ? 0.0f : s[i];
      acc = __fadd_rn(acc, __fmul_rn(q[i], sv));
    }
  }
  if (active) scores[c] = __fmul_rn(acc, scale);
}

// ---------------------------------------------------------------------------
// 1b. Certified scoring (the fast path).
//
// The sequential chain above is latency-bound (4096 dependent adds per page).
// Instead, each page gets one wave that forms the same fp32 products
// p_i = fl(q_i*s_i), sums them in double, and bounds how far the reference's
// sequential fp32 sum can be from that sum:
//   acc_i = fl(acc_{i-1} + p_i)  =>  |acc_n - S| <= u * sum_i |T_i| / (1 - n u)
// with S = sum p_i, T_i the exact prefix sums and u = 2^-24 (plus 2^-150 per
// step for subnormal results).  The page's score interval
// [fl(lo*scale), fl(hi*scale)] (lo/hi rounded outward to float) provably
// contains the reference score, because fl(x*scale) is monotone in x.
// At E = 4096 the fused step's float score passes (ScorePagesKernel in
// fused_step.hip) take this role; the kernel below serves the other E.
//
// Bound by the summary rows (4*E bytes a page against about 11 fp64 and 40
// other instructions per 256 products).  A row of 256 products is one float4
// per lane, so every load reads 1 KiB contiguously (a block of E/64
// consecutive products per lane, read one at a time, took 94 us for the 40 MB
// of 32 requests of 8 x 128 heads, about 300 pages each; this form
// 15 us).  Prefix sums: within the float4, then a wave scan of the lanes'
// sums, then the rows' totals one after the other; on any product's path at
// most 3 + 6 + E/256 + 2 double additions, far below the n roundings that
// WriteBounds allows for.  A wave takes `per_wave` pages of its request: their
// ids and token counts load once, lane i holding page i's, the next kRows rows
// load while this one's are summed, and page i's sums end in lane i, so the
// interval arithmetic runs once for all of them.  The query is staged in LDS
// up to kQueryLds bytes.
// ---------------------------------------------------------------------------
constexpr int kBoundWaves = 4;
constexpr int kBoundRows = 4;  // rows of 256 products in flight
constexpr size_t kBoundQueryLds = 64 * 1024;

// Any E that is a multiple of 64 (the last row may be part empty).  kRows = 1:
// E <= 256, one row, whose part of the query stays in each lane's registers (64
// requests of 250 pages of one 64-dim head: the step 23.5 us, 25.1 with four rows
// in flight and the query in LDS).
template <bool kQueryLds, int kRows>
__global__ __launch_bounds__(kBoundWaves * kWave) void ScoreBoundGenericKernel(
    const float* __restrict__ queries, const float* __restrict__ summaries,
    const int* __restrict__ token_counts, int capacity, const int* __restrict__ cand_offsets,
    const int* __restrict__ cand_ids, int total, int per_wave, int E, float scale,
    float* __restrict__ mid_out, float* __restrict__ lo_out, float* __restrict__ hi_out,
    FailReport fail) {
  extern __shared__ float4 q_lds[];
  const int r = blockIdx.y;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int groups = E / 4;  // float4 groups
  const float4* __restrict__ q4 =
      reinterpret_cast<const float4*>(queries + static_cast<size_t>(r) * E);
  int begin, n;
  const bool ok = RequestRange(cand_offsets, r, total, fail, &begin, &n);
  const int first = (static_cast<int>(blockIdx.x) * kBoundWaves + wave) * per_wave;
  if (!ok || static_cast<int>(blockIdx.x) * kBoundWaves * per_wave >= n) return;
  if constexpr (kQueryLds) {
    for (int i = threadIdx.x; i < groups; i += kBoundWaves * kWave) q_lds[i] = q4[i];
  }
  const int pages = n - first < per_wave ? n - first : per_wave;  // <= kWave
  // Lane i: page i of this wave; -1 (an id outside the pool, reported, or a
  // page holding no tokens) scores as an all-zero summary.
  int my_page = -1;
  if (lane < pages) {
    const int id = cand_ids[begin + first + lane];
    if (!InPool(id, capacity)) {
      ReportFailure(fail, kFailPageId);
    } else if (token_counts[id] != 0) {
      my_page = id;
    }
  }
  if constexpr (kQueryLds) __syncthreads();
  if (pages <= 0) return;
  const int rows = (groups + kWave - 1) / kWave;
  const int steps = kRows == 1 ? 1 : (rows + kRows - 1) / kRows;
  float4 only = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if constexpr (kRows == 1) {
    if (lane < groups) only = q4[lane];
  }
  float4 next[kRows];
  auto load = [&](int i, int step) {
    const int page = __builtin_amdgcn_readlane(my_page, i);
    const float4* s4 = reinterpret_cast<const float4*>(
        summaries + static_cast<size_t>(page < 0 ? 0 : page) * E);
#pragma unroll
    for (int u = 0; u < kRows; ++u) {
      const int g = (step * kRows + u) * kWave + lane;
      next[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (page >= 0 && g < groups) next[u] = s4[g];
    }
  };
  double my_sum = 0.0, my_prefix = 0.0, my_abs = 0.0;
  double carry = 0.0, abs_prefix = 0.0, abs_p = 0.0;
  load(0, 0);
  int i = 0, step = 0;
  for (int unit = 0; unit < pages * steps; ++unit) {
    float4 sv[kRows];
#pragma unroll
    for (int u = 0; u < kRows; ++u) sv[u] = next[u];
    const bool last_step = step + 1 == steps;
    const int ni = last_step ? i + 1 : i;
    const int nstep = last_step ? 0 : step + 1;
    if (ni < pages) load(ni, nstep);
#pragma unroll
    for (int u = 0; u < kRows; ++u) {
      const int row = step * kRows + u;
      if (kRows > 1 && row >= rows) break;
      const int g = row * kWave + lane;
      float4 qv = only;
      if (kRows > 1 && g < groups) {
        if constexpr (kQueryLds) {
          qv = q_lds[g];
        } else {
          qv = q4[g];
        }
      }
      const double p0 = static_cast<double>(__fmul_rn(qv.x, sv[u].x));
      const double p1 = static_cast<double>(__fmul_rn(qv.y, sv[u].y));
      const double p2 = static_cast<double>(__fmul_rn(qv.z, sv[u].z));
      const double p3 = static_cast<double>(__fmul_rn(qv.w, sv[u].w));
      const double l1 = p0 + p1;
      const double l2 = l1 + p2;
      const double l3 = l2 + p3;
      abs_p += (fabs(p0) + fabs(p1)) + (fabs(p2) + fabs(p3));
      const double incl = WaveInclusiveScanD(l3);
      // The prefix before this lane's group: exactly the lane below's scan.
      const double start = carry + DppMoveD<kWaveShr1>(incl);
      // (an empty group past E adds no prefix)
      if (g < groups) {
        abs_prefix += (fabs(start + p0) + fabs(start + l1)) +
                      (fabs(start + l2) + fabs(start + l3));
      }
      carry += ReadLaneD(incl, kWave - 1);
    }
    if (last_step) {
      const double tp = WaveSum(abs_prefix);
      const double ta = WaveSum(abs_p);
      if (lane == i) {
        my_sum = carry;
        my_prefix = tp;
        my_abs = ta;
      }
      carry = 0.0;
      abs_prefix = 0.0;
      abs_p = 0.0;
    }
    i = ni;
    step = nstep;
  }
  if (lane < pages) {
    WriteBounds(my_sum, my_prefix, my_abs, E, scale, mid_out, lo_out, hi_out,
                begin + first + lane);
  }
}

// ---------------------------------------------------------------------------
// 2. Top-k select.
//
// Each candidate becomes one 64-bit key whose unsigned order is the
// reference's comparator: high word = order-preserving image of the score
// (-0.0 folded onto +0.0, since the reference compares with ==), low word =
// ~page_id so that a smaller id wins a tie.  One workgroup bitonic-sorts a
// request's keys descending in LDS and emits the first min(k, n) ids.
// ---------------------------------------------------------------------------
constexpr int kSelectMaxKeys = 8192;  // 64 KiB of LDS

__global__ __launch_bounds__(256) void SelectTopKKernel(
    const float* __restrict__ scores, const int* __restrict__ cand_offsets,
    const int* __restrict__ cand_ids, int total, int max_candidates, int top_k,
    int* __restrict__ selected, int* __restrict__ counts, bool undecided_only, FailReport fail) {
  extern __shared__ uint64_t keys[];
  const int r = blockIdx.x;
  if (undecided_only && counts[r] >= 0) return;
  int begin, n;
  RequestRange(cand_offsets, r, total, fail, &begin, &n);
  if (n > max_candidates) {
    // The launch (LDS, score grid) was sized for max_candidates.
    if (threadIdx.x == 0) ReportFailure(fail, kFailShape);
    n = 0;
  }
  const int kk = top_k <= 0 ? 0 : (top_k < n ? top_k : n);
  if (kk == 0) {
    if (threadIdx.x == 0) counts[r] = 0;
    return;
  }
  int m = 1;
  int log_m = 0;
  while (m < n) {
    m <<= 1;
    ++log_m;
  }
  for (int i = threadIdx.x; i < m; i += blockDim.x) {
    keys[i] = i < n ? SelectKey(scores[begin + i], cand_ids[begin + i]) : 0ull;
  }
  __syncthreads();
  const int half = m >> 1;
  for (int log_size = 1; log_size <= log_m; ++log_size) {
    const int size = 1 << log_size;
    for (int log_stride = log_size - 1; log_stride >= 0; --log_stride) {
      const int stride = 1 << log_stride;
      for (int i = threadIdx.x; i < half; i += blockDim.x) {
        const int lo = ((i >> log_stride) << (log_stride + 1)) | (i & (stride - 1));
        const int hi = lo + stride;
        const bool descending = (lo & size) == 0;
        const uint64_t a = keys[lo];
        const uint64_t b = keys[hi];
        if ((a < b) == descending) {
          keys[lo] = b;
          keys[hi] = a;
        }
      }
      __syncthreads();
    }
  }
  int* out = selected + static_cast<size_t>(r) * top_k;
  for (int i = threadIdx.x; i < kk; i += blockDim.x) out[i] = KeyPage(keys[i]);
  if (threadIdx.x == 0) counts[r] = kk;
}

// ---------------------------------------------------------------------------
// 2b. Certified top-k select (257 to 8192 candidates per request; up to 256:
// SelectCertifiedRankKernel below).
//
// Candidates are ordered by (interval midpoint desc, id asc).  With T the
// first k, a candidate needs its exact score only if its interval overlaps
// another relevant one: an outsider whose hi reaches min(lo over T), or a
// member of T whose interval meets an outsider's or another member's.  Every
// other comparison is already decided by disjoint intervals, so replacing the
// open candidates' keys by their exact scores and sorting again yields the
// reference order exactly.  Before that the open candidates get refined
// intervals (RefineScores), which usually decide them.  Exact scores come from
// the reference's sequential chain (RescoreChains: the lanes of wave 0 run the
// dependent adds of up to 32 pages while the other waves form the next stretch
// of products).
//
// One request is one workgroup's chain of loads, radix rounds, sort and
// certification, so it is latency-bound.  A candidate's key and interval stay
// in the registers of one thread (candidate i in thread i mod 1024) until the
// set that can still be selected is in LDS, and order and certification then
// only see that set, several threads per element.  8192 candidates of one
// request take 14.6 us with one selected; with 64, whose order some 8 pages'
// intervals leave open, 24 us (42 us with one thread per member in the sort and
// the certification and the radix rounds run again after the refinement).
// Beyond 2048 candidates this replaces exact chains for every page (154 us for
// 4 requests of up to 8192 pages) and a bitonic sort of them (165 us): that
// step took 363 us and takes 137.  Up to 2048 candidates it replaces a select
// that kept every candidate in LDS and gave each member one thread (32 requests
// of 8 x 128 heads, 300 pages each: the step 50 us, 45.5 with this select alone
// changed; the wide step of one request of 2048 pages, 64 selected: 71 us, 59).
//
// Beyond 2048 candidates LDS holds kLargeMaxK members and kLargeMaxOpen open
// candidates: a request with more open (equal pages, a zero query) is left
// undecided, counts[r] = kUndecided, for the exact score and select kernels
// that the launch enqueues after this one and that return at once for every
// other request; chains here take 25 us per 32 candidates.
// ---------------------------------------------------------------------------
constexpr int kCertMaxKeys = 2048;    // candidates per request with no bound on the open ones
constexpr int kSelRescoreGroup = 32;  // exact chains per rescore group (lanes of wave 0)
constexpr int kSelThreads = 1024;

// One wave: the bucket of a 256-bin histogram that holds the need-th largest
// key: *s_prefix = prefix with the bucket's 8 bits appended, *s_need the
// members it still owes, *s_all whether it owes all its keys.
__device__ __forceinline__ void RadixBucket(const int* hist, uint64_t prefix, int need,
                                            unsigned long long* s_prefix, int* s_need,
                                            int* s_all) {
  const int lane = threadIdx.x & (kWave - 1);
  // Lane l holds bins 4l .. 4l+3; suffix sums from the top bin down find
  // the bucket b with sum(bins > b) < need <= sum(bins >= b).
  const int b0 = 4 * lane;
  const int c3 = hist[b0 + 3], c2 = hist[b0 + 2], c1 = hist[b0 + 1], c0 = hist[b0];
  int suffix = c0 + c1 + c2 + c3;  // becomes the sum over lanes >= l
  for (int o = 1; o < kWave; o <<= 1) {
    const int other = __shfl_down(suffix, o, kWave);
    if (lane + o < kWave) suffix += other;
  }
  int above = __shfl_down(suffix, 1, kWave);  // sum over lanes > l
  if (lane == kWave - 1) above = 0;
  if (suffix >= need && above < need) {
    int b = b0 + 3;
    int count = c3;
    if (above + c3 < need) { above += c3; b = b0 + 2; count = c2;
      if (above + c2 < need) { above += c2; b = b0 + 1; count = c1;
        if (above + c1 < need) { above += c1; b = b0; count = c0; } } }
    *s_prefix = (static_cast<unsigned long long>(prefix) << 8) | static_cast<unsigned>(b);
    *s_need = need - above;
    *s_all = count == need - above;
  }
}

// A tagged word once it carries `tag` (spin_limit polls, sleeping between),
// or false.
__device__ __forceinline__ bool AwaitTagged(unsigned long long* p, unsigned tag,
                                            unsigned spin_limit, unsigned long long* out) {
  unsigned long long w = LoadWord(p);
  for (unsigned i = 0; static_cast<unsigned>(w >> 32) != tag; ++i) {
    if (i >= spin_limit) return false;
    __builtin_amdgcn_s_sleep(1);
    w = LoadWord(p);
  }
  *out = w;
  return true;
}

constexpr int kLargeMaxKeys = 8192;
constexpr int kLargeMaxK = 1024;
constexpr int kLargeMaxOpen = 128;
constexpr int kUndecided = -1;
// Flagged pages that the helper workgroups refine: fewer are as quick in the
// selecting workgroup (no exchange), more go to the exact chains.
constexpr int kAssistLeastPages = 3;
constexpr int kAssistMaxPages = 64;
constexpr int kAssistMaxHelpers = 32;
constexpr int kAssistLeastCandidates = 256;  // room for the words
static_assert(1 + 4 * kAssistMaxPages <= 3 * kAssistLeastCandidates, "the words fit");
static_assert(3 * kAssistMaxPages <= kSelThreads, "a thread per word");

// The candidates that can still be in the top kk: the members (the kk largest
// midpoints) and the outsiders whose interval reaches the members' smallest
// lower bound.  Every other outsider's score lies below every member's, so it
// is out whatever the open intervals hide.
template <int kSet>
struct CertSet {
  uint64_t key[kSet];
  int c[kSet];  // candidate
  float lo[kSet], hi[kSet];
};
// The LDS of one request's certified select.  kSet: candidates the set holds;
// kOpen: how many may be open.
template <int kSet_, int kOpen_>
struct CertSharedT {
  static constexpr int kSet = kSet_;
  static constexpr int kOpen = kOpen_;
  CertSet<kSet> a, b;  // one is sorted into the other
  int open[kOpen];     // positions whose order is open
  int page_c[kAssistMaxPages];  // a helper's pages
  float r_mid[kAssistMaxPages], r_lo[kAssistMaxPages], r_hi[kAssistMaxPages];
  int hist[256];
  float red[kSelThreads / kWave];
  unsigned long long prefix;
  int need, all, count, tie, nopen, bad;
  alignas(16) float tile[RescoreFloats<kSelRescoreGroup>()];
};
using CertShared = CertSharedT<kCertMaxKeys, kCertMaxKeys>;
using CertSharedLarge = CertSharedT<kLargeMaxK + kLargeMaxOpen, kLargeMaxOpen>;

// Threads per element of a pass over the set: 1 << shift, 4 to 16.  The loops
// below compare every pair, about ten instructions each on all four SIMDs, so
// what matters is that no wave runs without elements and that the reads need no
// bounds test: sets beyond 256 take several passes of 256, a wave past the last
// element skips its loop, and four reads at a time are whole.  The select of 512
// of 520 candidates takes 100 us (111 with a test per read), of 513 of 1040
// 106 (170 with one thread an element and every wave in the loop).
__device__ __forceinline__ int SetShift(int count) {
  int shift = 4;
  while (shift > 2 && (count << shift) > kSelThreads) --shift;
  return shift;
}
// Whether this wave has an element in the pass from element `base` on.
__device__ __forceinline__ bool SetWaveBusy(int base, int shift, int count) {
  const int wave_first = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x));
  return base + (wave_first >> shift) < count;
}

// from, sorted by key (descending; equal keys by position), into to: ranks by
// counting, `parts` threads per element.  Ends with a barrier.
template <class Set>
__device__ __forceinline__ void SortSet(const Set& from, Set& to, int count) {
  const int shift = SetShift(count);
  const int parts = 1 << shift;
  const int part = threadIdx.x & (parts - 1);
  for (int base = 0; base < count; base += kSelThreads >> shift) {
    if (!SetWaveBusy(base, shift, count)) break;
    const int t = base + (static_cast<int>(threadIdx.x) >> shift);
    const uint64_t k = t < count ? from.key[t] : 0ull;
    int rank = 0;
    int u = part;
    for (; u + 3 * parts < count; u += 4 * parts) {
      uint64_t ku[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) ku[v] = from.key[u + v * parts];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        rank += (ku[v] > k) | ((ku[v] == k) & (u + v * parts < t));
      }
    }
    for (; u < count; u += parts) {
      const uint64_t ku = from.key[u];
      rank += (ku > k) | ((ku == k) & (u < t));
    }
    for (int o = 1; o < parts; o <<= 1) rank += __shfl_xor(rank, o, kWave);
    if (t < count && part == 0) {
      to.key[rank] = k;
      to.c[rank] = from.c[t];
      to.lo[rank] = from.lo[t];
      to.hi[rank] = from.hi[t];
    }
  }
  __syncthreads();
}

// The positions of the sorted set whose order among the first kk, or across
// that line, its intervals leave open: a position below kk whose interval
// meets any other's, and one from kk on whose interval meets a member's.
// Appends them to sh.open (sh.nopen counts all of them).  Ends with a barrier.
template <class Shared, class Set>
__device__ __forceinline__ void CertifySet(Shared& sh, const Set& set, int count, int kk) {
  const int shift = SetShift(count);
  const int parts = 1 << shift;
  const int part = threadIdx.x & (parts - 1);
  for (int base = 0; base < count; base += kSelThreads >> shift) {
    if (!SetWaveBusy(base, shift, count)) break;
    const int t = base + (static_cast<int>(threadIdx.x) >> shift);
    const bool in = t < count;
    const float l = in ? set.lo[t] : INFINITY;
    const float h = in ? set.hi[t] : -INFINITY;
    const int others = t < kk ? count : kk;
    int open = 0;
    int u = part;
    for (; u + 3 * parts < others; u += 4 * parts) {
      float lu[4], hu[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        lu[v] = set.lo[u + v * parts];
        hu[v] = set.hi[u + v * parts];
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        open |= (u + v * parts != t) & (l <= hu[v]) & (lu[v] <= h);
      }
    }
    for (; u < others; u += parts) {
      open |= (u != t) & (l <= set.hi[u]) & (set.lo[u] <= h);
    }
    for (int o = 1; o < parts; o <<= 1) open |= __shfl_xor(open, o, kWave);
    if (in && open != 0 && part == 0) {
      const int pos = atomicAdd(&sh.nopen, 1);
      if (pos < Shared::kOpen) sh.open[pos] = t;
    }
  }
  __syncthreads();
}

// A helper workgroup of a large request's select: once the request's
// workgroup has published its flagged candidates, refines every helpers-th of
// them from its first-pass interval and publishes the result.  One workgroup
// refines a page in 4-6 us with half its waves, and refining 8 to 64 pages in
// the selecting workgroup, or running their exact chains (25 us a group of 32),
// is what its time went to while the rest of the chip stood idle.
template <class Shared>
__device__ __forceinline__ void AssistSelect(Shared& sh, const SelectAssist& assist,
                                            unsigned long long* words, int index,
                                            const float* __restrict__ lo,
                                            const float* __restrict__ hi,
                                            const float* __restrict__ q,
                                            const float* __restrict__ summaries,
                                            const int* __restrict__ token_counts, int capacity,
                                            const int* __restrict__ cand, int n, int E,
                                            float scale) {
  const int tid = threadIdx.x;
  if (tid == 0) {
    unsigned long long w = 0;
    const bool ok = AwaitTagged(words, assist.WaitTag(), assist.spin_limit, &w);
    const int pages = ok ? static_cast<int>(static_cast<uint32_t>(w)) : 0;
    sh.nopen = pages <= kAssistMaxPages ? pages : 0;
    sh.all = 1;
  }
  __syncthreads();
  const int pages = sh.nopen;
  const int mine = index < pages ? (pages - index + assist.helpers - 1) / assist.helpers : 0;
  if (mine == 0) return;
  if (tid < mine) {
    unsigned long long w = 0;
    const bool ok = AwaitTagged(words + 1 + index + tid * assist.helpers, assist.WaitTag(),
                                assist.spin_limit, &w);
    const int c = static_cast<int>(static_cast<uint32_t>(w));
    if (!ok || c < 0 || c >= n) {
      sh.all = 0;
    } else {
      sh.page_c[tid] = c;
      sh.r_lo[tid] = lo[c];
      sh.r_hi[tid] = hi[c];
    }
  }
  __syncthreads();
  if (sh.all == 0) return;  // (the request's workgroup gives up waiting, too)
  RefineScores<kSelThreads>(
      mine,
      [&](int f) -> const float* {
        const int pg = cand[sh.page_c[f]];
        const bool live = InPool(pg, capacity) && token_counts[pg] != 0;
        return live ? summaries + static_cast<size_t>(pg) * E : nullptr;
      },
      [&](int f) { return dsd_refine::FirstPassBound(sh.r_lo[f], sh.r_hi[f], scale, E); },
      [&](int f, float m, float l, float h) {
        unsigned long long* to =
            words + 1 + kAssistMaxPages + 3 * (index + f * assist.helpers);
        PutTagged(to, assist.epoch, __float_as_uint(m));
        PutTagged(to + 1, assist.epoch, __float_as_uint(l));
        PutTagged(to + 2, assist.epoch, __float_as_uint(h));
      },
      q, E, scale, reinterpret_cast<double*>(sh.tile));
}

// Request r's certified top-k (up to PER * kSelThreads candidates, the whole
// workgroup of kSelThreads threads).  load(c, &mid, &lo, &hi) gives candidate
// c's first-pass interval (c indexes the batch's CSR); with kPolled it may
// report that an interval never became readable (false), and the request
// then selects nothing (kFailWait).  emit(i, page) writes member i of the
// selection (rank order), emit_count(kk) the count (or kUndecided); emit_count
// runs once, in thread 0, after the emits.  words: the request's assist words,
// or null.
template <int PER, bool kPolled, class Shared, class Load, class Emit, class EmitCount>
__device__ __forceinline__ void SelectCertifiedRequest(
    Shared& sh, int begin, int n, int kk, Load load, Emit emit, EmitCount emit_count,
    const float* __restrict__ q, const float* __restrict__ summaries,
    const int* __restrict__ token_counts, int capacity, const int* __restrict__ cand, int E,
    float scale, int* __restrict__ exact_pages, const SelectAssist& assist,
    unsigned long long* words, FailReport fail) {
  static_assert(PER <= 32, "a member bit per candidate");
  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = tid / kWave;
  if (tid == 0) {
    sh.count = 0;
    sh.tie = 0;
    sh.nopen = 0;
    sh.bad = 0;
  }
  if constexpr (kPolled) __syncthreads();
  uint64_t key[PER];
  float clo[PER], chi[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int i = tid + kSelThreads * j;
    key[j] = 0;
    clo[j] = INFINITY;
    chi[j] = -INFINITY;
    if (i < n) {
      float m;
      if (!load(begin + i, &m, &clo[j], &chi[j])) sh.bad = 1;
      key[j] = SelectKey(m, cand[i]);
    }
  }
  if constexpr (kPolled) {
    __syncthreads();
    if (sh.bad != 0) {
      if (tid == 0) {
        ReportFailure(fail, kFailWait);
        emit_count(0);
      }
      return;
    }
  }
  // 1. The kk-th largest key, 8 bits a round.
  uint64_t prefix = 0;
  int need = kk;
  int shift = 56;
  bool all = false;
  for (int round = 0; round < 8 && !all; ++round) {
    shift = 56 - 8 * round;
    if (tid < 256) sh.hist[tid] = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const bool in = tid + kSelThreads * j < n &&
                      (round == 0 || (key[j] >> (shift + 8)) == prefix);
      if (in) atomicAdd(&sh.hist[static_cast<int>((key[j] >> shift) & 255u)], 1);
    }
    __syncthreads();
    if (wave == 0) {
      RadixBucket(sh.hist, prefix, need, &sh.prefix, &sh.need, &sh.all);
    }
    __syncthreads();
    prefix = sh.prefix;
    need = sh.need;
    all = sh.all != 0;
  }
  // 2. The set: the members, then the outsiders that reach them.
  unsigned members = 0;
  float my_min = INFINITY;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int i = tid + kSelThreads * j;
    const uint64_t top = key[j] >> shift;
    bool in = i < n && top > prefix;
    if (i < n && top == prefix) in = all || atomicAdd(&sh.tie, 1) < need;
    if (in) {
      members |= 1u << j;
      const int pos = atomicAdd(&sh.count, 1);
      sh.a.key[pos] = key[j];
      sh.a.c[pos] = i;
      sh.a.lo[pos] = clo[j];
      sh.a.hi[pos] = chi[j];
      my_min = fminf(my_min, clo[j]);
    }
  }
  for (int o = 1; o < kWave; o <<= 1) my_min = fminf(my_min, __shfl_xor(my_min, o, kWave));
  if (lane == 0) sh.red[wave] = my_min;
  __syncthreads();
  float min_t_lo = INFINITY;
  for (int w = 0; w < kSelThreads / kWave; ++w) min_t_lo = fminf(min_t_lo, sh.red[w]);
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int i = tid + kSelThreads * j;
    if (i < n && !((members >> j) & 1u) && chi[j] >= min_t_lo) {
      const int pos = atomicAdd(&sh.count, 1);
      if (pos < Shared::kSet && pos < kk + Shared::kOpen) {
        sh.a.key[pos] = key[j];
        sh.a.c[pos] = i;
        sh.a.lo[pos] = clo[j];
        sh.a.hi[pos] = chi[j];
      }
    }
  }
  __syncthreads();
  const int count = sh.count;
  const bool too_many = count > Shared::kSet || count > kk + Shared::kOpen;
  // 3. Their order, and what the first-pass intervals leave open.  (A member
  //    that meets an outsider meets one of the set.)
  if (!too_many) {
    SortSet(sh.a, sh.b, count);
    CertifySet(sh, sh.b, count, kk);
  }
  int nopen = too_many ? Shared::kOpen + 1 : sh.nopen;
  const bool refine = E % 256 == 0 && nopen > 0;
  const bool share =
      refine && words != nullptr && nopen >= kAssistLeastPages && nopen <= kAssistMaxPages;
  if (words != nullptr) {
    // The helpers' share (0: they leave).
    if (tid < (share ? nopen : 0)) {
      PutTagged(words + 1 + tid, assist.epoch, static_cast<uint32_t>(sh.b.c[sh.open[tid]]));
    }
    if (tid == 0) {
      PutTagged(words, assist.epoch, static_cast<uint32_t>(share ? nopen : 0));
    }
  }
  // (the exact kernels then chain every candidate)
  auto defer = [&] {
    if (tid != 0) return;
    if (exact_pages != nullptr) atomicAdd(exact_pages, n);
    emit_count(kUndecided);
  };
  if (nopen > Shared::kOpen) {
    defer();
    return;
  }
  auto* order = &sh.b;
  if (share || (refine && RefineWorthwhile<kSelThreads>(nopen))) {
    // 4. Refined intervals of the open positions (sh.r_*), by the helpers
    //    or here, and the set's order again.  A wait that gives up leaves the
    //    first-pass intervals, which are sound, to the exact chains.
    if (tid == 0) sh.all = 1;
    __syncthreads();
    if (share) {
      // Thread 3f + x: word x of open position f's interval.
      if (tid < 3 * nopen) {
        unsigned long long w = 0;
        if (AwaitTagged(words + 1 + kAssistMaxPages + tid, assist.WaitTag(), assist.spin_limit,
                        &w)) {
          float* to = tid % 3 == 0 ? sh.r_mid : (tid % 3 == 1 ? sh.r_lo : sh.r_hi);
          to[tid / 3] = __uint_as_float(static_cast<uint32_t>(w));
        } else {
          sh.all = 0;
        }
      }
      __syncthreads();
    } else {
      RefineScores<kSelThreads>(
          nopen,
          [&](int f) -> const float* {
            const int pg = cand[sh.b.c[sh.open[f]]];
            const bool live = InPool(pg, capacity) && token_counts[pg] != 0;
            return live ? summaries + static_cast<size_t>(pg) * E : nullptr;
          },
          [&](int f) {
            const int t = sh.open[f];
            return dsd_refine::FirstPassBound(sh.b.lo[t], sh.b.hi[t], scale, E);
          },
          [&](int f, float m, float l, float h) {
            sh.r_mid[f] = m;
            sh.r_lo[f] = l;
            sh.r_hi[f] = h;
          },
          q, E, scale, reinterpret_cast<double*>(sh.tile));
    }
    if (sh.all != 0) {
      if (tid < nopen) {
        const int t = sh.open[tid];
        sh.b.key[t] = SelectKey(sh.r_mid[tid], cand[sh.b.c[t]]);
        sh.b.lo[t] = sh.r_lo[tid];
        sh.b.hi[t] = sh.r_hi[tid];
      }
      if (tid == 0) sh.nopen = 0;
      __syncthreads();
      SortSet(sh.b, sh.a, count);
      CertifySet(sh, sh.a, count, kk);
      order = &sh.a;
      nopen = sh.nopen;
      if (nopen > Shared::kOpen) {
        defer();
        return;
      }
    }
  }
  if (nopen > 0) {
    // 5. Exact chains for what is still open, and the order once more.
    if (tid == 0 && exact_pages != nullptr) atomicAdd(exact_pages, nopen);
    auto& set = *order;
    RescoreChains<kSelRescoreGroup, kSelThreads>(
        nopen, [&](int f) { return cand[set.c[sh.open[f]]]; },
        [&](int f, float score) {
          const int t = sh.open[f];
          set.key[t] = SelectKey(score, cand[set.c[t]]);
        },
        q, summaries, token_counts, capacity, E, scale, sh.tile);
    auto* other = order == &sh.a ? &sh.b : &sh.a;
    SortSet(set, *other, count);
    order = other;
  }
  for (int i = tid; i < kk; i += kSelThreads) emit(i, KeyPage(order->key[i]));
  if constexpr (kPolled) __syncthreads();  // every member out before the count
  if (tid == 0) emit_count(kk);
}

// Request r's candidates and how many to select; none (reported) when there
// are more than the score kernel covered or the select holds.
__device__ __forceinline__ int SelectRange(const int* cand_offsets, int r, int total,
                                           int max_candidates, int most, int top_k,
                                           const FailReport& fail, bool report, int* begin,
                                           int* n) {
  RequestRange(cand_offsets, r, total, report ? fail : FailReport{}, begin, n);
  if (*n > max_candidates || *n > most) {
    if (report && threadIdx.x == 0) ReportFailure(fail, kFailShape);
    *n = 0;
  }
  return top_k <= 0 ? 0 : (top_k < *n ? top_k : *n);
}

// Workgroup r < batch: request r's select; the others its helpers.
template <int PER, class Shared>
__global__ __launch_bounds__(kSelThreads) void SelectCertifiedKernel(
    const float* __restrict__ mid, const float* __restrict__ lo,
    const float* __restrict__ hi, const float* __restrict__ queries,
    const float* __restrict__ summaries, const int* __restrict__ token_counts, int capacity,
    const int* __restrict__ cand_offsets, const int* __restrict__ cand_ids, int batch, int total,
    int max_candidates, int E, float scale, int top_k, int* __restrict__ selected,
    int* __restrict__ counts, int* __restrict__ exact_pages, SelectAssist assist,
    FailReport fail) {
  __shared__ Shared sh;
  const bool helper = static_cast<int>(blockIdx.x) >= batch;
  const int r = static_cast<int>(blockIdx.x) % batch;
  int begin, n;
  const int kk = SelectRange(cand_offsets, r, total, max_candidates, PER * kSelThreads, top_k,
                             fail, !helper, &begin, &n);
  const int* cand = cand_ids + begin;
  const float* q = queries + static_cast<size_t>(r) * E;
  // The request's assist words lie in its candidates' publication words
  // (idle in this step form): [0] the pages to refine, [1 ..] which
  // candidates, then three words of interval per page.
  unsigned long long* words = assist.helpers > 0 && n > kAssistLeastCandidates
                                  ? assist.words + 3 * static_cast<size_t>(begin)
                                  : nullptr;
  if (helper) {
    if (kk > 0 && words != nullptr) {
      AssistSelect(sh, assist, words, (static_cast<int>(blockIdx.x) - batch) / batch, lo + begin,
                   hi + begin, q, summaries, token_counts, capacity, cand, n, E, scale);
    }
    return;
  }
  if (kk == 0) {
    if (threadIdx.x == 0) counts[r] = 0;
    return;
  }
  int* out = selected + static_cast<size_t>(r) * top_k;
  SelectCertifiedRequest<PER, false>(
      sh, begin, n, kk,
      [&](int c, float* m, float* l, float* h) {
        *m = mid[c];
        *l = lo[c];
        *h = hi[c];
        return true;
      },
      [&](int i, int page) { out[i] = page; }, [&](int count) { counts[r] = count; }, q,
      summaries, token_counts, capacity, cand, E, scale, exact_pages, assist, words, fail);
}

// Certified select for up to 256 candidates per request: thread i owns
// candidate i and finds its rank by counting larger keys (broadcast LDS reads,
// no barrier chain), ties broken by position so ranks are distinct.
constexpr int kRankMax = 256;

__global__ __launch_bounds__(kRankMax) void SelectCertifiedRankKernel(
    const float* __restrict__ mid, const float* __restrict__ lo,
    const float* __restrict__ hi, const float* __restrict__ queries,
    const float* __restrict__ summaries, const int* __restrict__ token_counts, int capacity,
    const int* __restrict__ cand_offsets, const int* __restrict__ cand_ids, int total,
    int max_candidates, int E, float scale, int top_k, int* __restrict__ selected,
    int* __restrict__ counts, int* __restrict__ exact_pages, FailReport fail) {
  __shared__ uint64_t s_key[kRankMax];
  __shared__ float s_lo[kRankMax];
  __shared__ float s_hi[kRankMax];
  __shared__ int s_top[kRankMax];
  __shared__ int s_flag[kRankMax];
  __shared__ float s_red[2][kRankMax / kWave];
  __shared__ int s_nflag;
  __shared__ __align__(16) float tile[RescoreFloats<kSelRescoreGroup>()];
  const int r = blockIdx.x;
  int begin, n;
  RequestRange(cand_offsets, r, total, fail, &begin, &n);
  if (n > max_candidates || n > kRankMax) {
    // Only max_candidates were scored (and this kernel holds kRankMax):
    // select nothing and report it.
    if (threadIdx.x == 0) ReportFailure(fail, kFailShape);
    n = 0;
  }
  const int kk = top_k <= 0 ? 0 : (top_k < n ? top_k : n);
  if (kk == 0) {
    if (threadIdx.x == 0) counts[r] = 0;
    return;
  }
  const int i = threadIdx.x;
  const bool active = i < n;
  if (active) {
    s_key[i] = SelectKey(mid[begin + i], cand_ids[begin + i]);
    s_lo[i] = lo[begin + i];
    s_hi[i] = hi[begin + i];
  }
  if (i == 0) s_nflag = 0;
  __syncthreads();
  // Keys are read 8 at a time (independent broadcast LDS reads in flight).
  auto rank_of = [&](int me) {
    const uint64_t key = s_key[me];
    int rank = 0;
    int j = 0;
    for (; j + 8 <= n; j += 8) {
      uint64_t kj[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) kj[u] = s_key[j + u];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        rank += (kj[u] > key || (kj[u] == key && j + u < me)) ? 1 : 0;
      }
    }
    for (; j < n; ++j) {
      const uint64_t kj = s_key[j];
      rank += (kj > key || (kj == key && j < me)) ? 1 : 0;
    }
    return rank;
  };
  const int wave = threadIdx.x / kWave;
  constexpr int nwaves = kRankMax / kWave;
  const int* cand = cand_ids + begin;
  int rank = n;
  int nflag = 0;
  // Pass 0 certifies with the score kernel's intervals; pages it leaves
  // open get refined intervals (RefineScores, several waves per page; E a
  // multiple of 256) and pass 1 certifies again.  What pass 1 leaves open
  // gets the exact chain.
  for (int pass = 0; pass < 2; ++pass) {
    rank = active ? rank_of(i) : n;
    if (active && rank < kk) s_top[rank] = i;
    float my_min = (active && rank < kk) ? s_lo[i] : INFINITY;
    float my_max = (active && rank >= kk) ? s_hi[i] : -INFINITY;
    for (int o = 1; o < kWave; o <<= 1) {
      my_min = fminf(my_min, __shfl_xor(my_min, o, kWave));
      my_max = fmaxf(my_max, __shfl_xor(my_max, o, kWave));
    }
    if ((threadIdx.x & (kWave - 1)) == 0) {
      s_red[0][wave] = my_min;
      s_red[1][wave] = my_max;
    }
    __syncthreads();
    float min_t_lo = INFINITY, max_o_hi = -INFINITY;
    for (int w = 0; w < nwaves; ++w) {
      min_t_lo = fminf(min_t_lo, s_red[0][w]);
      max_o_hi = fmaxf(max_o_hi, s_red[1][w]);
    }
    if (active) {
      const float l = s_lo[i];
      const float h = s_hi[i];
      bool flag;
      if (rank >= kk) {
        flag = h >= min_t_lo;
      } else {
        flag = l <= max_o_hi;
        for (int j = 0; j < kk && !flag; ++j) {
          if (j == rank) continue;
          const int c2 = s_top[j];
          flag = l <= s_hi[c2] && s_lo[c2] <= h;
        }
      }
      if (flag) s_flag[atomicAdd(&s_nflag, 1)] = i;
    }
    __syncthreads();
    nflag = s_nflag;
    if (nflag == 0 || pass == 1 || E % 256 != 0 || !RefineWorthwhile<kRankMax>(nflag)) break;
    RefineScores<kRankMax>(
        nflag,
        [&](int f) -> const float* {
          const int pg = cand[s_flag[f]];
          const bool live = pg >= 0 && pg < capacity && token_counts[pg] != 0;
          return live ? summaries + static_cast<size_t>(pg) * E : nullptr;
        },
        [&](int f) {
          const int c = s_flag[f];
          return dsd_refine::FirstPassBound(s_lo[c], s_hi[c], scale, E);
        },
        [&](int f, float m, float l, float h) {
          const int c = s_flag[f];
          // LDS only (see SelectCertifiedKernel).
          s_key[c] = SelectKey(m, cand[c]);
          s_lo[c] = l;
          s_hi[c] = h;
        },
        queries + static_cast<size_t>(r) * E, E, scale, reinterpret_cast<double*>(tile));
    if (i == 0) s_nflag = 0;
    __syncthreads();
  }
  if (nflag > 0) {
    if (threadIdx.x == 0 && exact_pages != nullptr) atomicAdd(exact_pages, nflag);
    RescoreChains<kSelRescoreGroup, kRankMax>(
        nflag, [&](int f) { return cand[s_flag[f]]; },
        [&](int f, float score) {
          const int c = s_flag[f];
          s_key[c] = SelectKey(score, cand[c]);
        },
        queries + static_cast<size_t>(r) * E, summaries, token_counts, capacity, E, scale, tile);
    rank = active ? rank_of(i) : n;
  }
  if (active && rank < kk) selected[static_cast<size_t>(r) * top_k + rank] = cand_ids[begin + i];
  if (threadIdx.x == 0) counts[r] = kk;
}

// ---------------------------------------------------------------------------
// 4. The wide step: the three-kernel step (E = 4096, head_dim 128, up to
// kCertMaxKeys candidates per request) in one launch.
//
// Items: score slices (request r, slice x: candidates [P*x, P*x + P), G
// slices per request) and attention items (request r, head h).  The
// workgroup that scores a request's last slice (an arrival counter per
// request) runs that request's certified select.  Every score slice comes
// before every attention item (WideItemOf with lag = batch): an attention
// item dispatched in the first round would hold its CU from the launch on
// while it waits for its select (at 32 requests of 2048 pages the step
// spanned 379 us with all slices first, 427-489 us with 4 to 16 requests'
// slices between a request's slices and its attention).  HBM streams K/V
// for the requests selected first while the others still score and select:
// the stages of different requests overlap instead of running one after
// another with HBM idle between them (reference: the score -> top-k ->
// attention sequence of src/cuda/sparse_batched_attention.cu:665-762 and
// its k > 16 path, :703-731).
//
// Tickets.  A workgroup takes the next item from a counter as it starts,
// and the grid holds half as many spare workgroups again, which find the
// items gone and leave.  Workgroup i goes to XCD i mod
// 8 and each XCD runs its own share of the grid: with items tied to
// workgroup ids, the XCDs whose CUs ran the selects (each holds its CU for
// about 47 us) finished up to 25 us after the others; with tickets an XCD
// that frees up early takes more items (config 3: 381 against 395 us per
// step; spares of 1 and 2 per item measured 383 and 388 us).
//
// Intervals, selected ids and counts cross workgroups as epoch-tagged
// words (score_slice.h): no fences.
//
// Every wait ends.  A score slice never waits; the select that follows a
// request's last slice waits only for interval words that the request's
// slices wrote before they arrived.  An attention item waits for its
// request's select, that is for score slices with lower tickets, which
// workgroups already running took: they finish without waiting, the last
// of them runs the select, and the select ends.  (Without tickets, the
// lowest-id attention item that waits has, on every XCD, only score slices
// and attention items that do not wait forever ahead of it in dispatch
// order, and the same follows.)  The polls are bounded anyway (kFailWait,
// zero outputs, never a hang).  The ticket and arrival counters come in two
// sets that launches use in turn; workgroup 0 of each launch zeroes the set
// the next launch will use (the previous launch used it and has finished),
// so no workgroup waits at the end to reset anything and a spare leaves
// after one load.
//
// A persistent form (one workgroup per CU taking items from a counter)
// spilled 188 bytes per lane: values the compiler hoisted out of the item
// loop stay live across all three item kinds.
// ---------------------------------------------------------------------------
constexpr int kWideStamps = 5;  // per item in timing mode
static_assert(kWideAttnWaves == kFWaves, "an attention item is a whole workgroup");

struct WideShared {
  union {
    ScoreShared score;
    CertShared cert;
    struct {
      AttnFastShared<kFWaves, 128> attn;
      int page[kCertMaxKeys];  // the item's selected pages
    };
  };
  int item;
  int last;
  int count;
  unsigned long long stamp[3];  // timing mode: start, select start and end
};

// Item i's kind (0 score slice, 1 attention), request and slice or head:
// request r's G slices, then (for r >= lag) request r - lag's Q heads,
// request by request; after the last request the remaining lag requests'
// heads.  (lag = batch: all slices, then all heads; DSD_WIDE_LAG.)
__device__ __forceinline__ int WideItemOf(int i, int batch, int G, int Q, int lag, int* r,
                                          int* sub) {
  const int head = lag * G;
  if (i < head) {
    *r = i / G;
    *sub = i - *r * G;
    return 0;
  }
  const int block = G + Q;
  const int j = (i - head) / block;
  if (j < batch - lag) {
    const int off = i - head - j * block;
    if (off < G) {
      *r = lag + j;
      *sub = off;
      return 0;
    }
    *r = j;
    *sub = off - G;
    return 1;
  }
  const int t = i - head - (batch - lag) * block;
  *r = batch - lag + t / Q;
  *sub = t - (t / Q) * Q;
  return 1;
}

// Item `item` of the step (WideItemOf), by the whole workgroup.
__device__ __forceinline__ void WideStepItem(const PoolView& pool, const WideArgs& w, int item,
                                             WideShared& sh) {
  const FusedArgs& a = w.a;
  const int stride = a.sel_stride;
  int item_r, item_sub;
  const int kind =
      WideItemOf(item, a.batch, w.groups, pool.num_heads, w.lag, &item_r, &item_sub);
  // Timing mode: thread 0's clocks (start, select start and end, end) and
  // the item kind, written out at the end.
  // (kept in LDS: a register would stay live across the whole item)
  if (a.stamps != nullptr && threadIdx.x == 0) {
    sh.stamp[0] = wall_clock64();
    sh.stamp[1] = 0;
    sh.stamp[2] = 0;
  }
  if (kind == 0) {
    const int r = item_r;
    const int x = item_sub;
    int begin, n;
    if (RequestRange(a.cand_offsets, r, a.total, x == 0 ? a.fail : FailReport{}, &begin, &n)) {
      const int c0 = x * w.pages_per_group;
      if (c0 < n) {
        const int c1 = n - c0 < w.pages_per_group ? n : c0 + w.pages_per_group;
        ScoreSlice<true>(pool, a, r, begin + c0, begin + c1, sh.score);
      }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      const unsigned prev = __hip_atomic_fetch_add(w.counters + 1 + r, 1u, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
      sh.last = prev == static_cast<unsigned>(w.groups - 1) ? 1 : 0;
    }
    __syncthreads();
    if (sh.last != 0) {
      if (a.stamps != nullptr && threadIdx.x == 0) sh.stamp[1] = wall_clock64();
      unsigned long long* sel = w.sel_rec + static_cast<size_t>(r) * stride;
      int* out = a.selected + static_cast<size_t>(r) * stride;
      int begin, n;
      const int kk = SelectRange(a.cand_offsets, r, a.total, a.max_candidates, kCertMaxKeys,
                                 a.top_k, a.fail, true, &begin, &n);
      auto emit_count = [&](int count) {
        a.counts[r] = count;
        PutTagged(w.cnt_rec + r, a.epoch, static_cast<uint32_t>(count));
      };
      if (kk == 0) {
        if (threadIdx.x == 0) emit_count(0);
      } else {
        SelectCertifiedRequest<kCertMaxKeys / kSelThreads, true>(
            sh.cert, begin, n, kk,
            [&](int c, float* m, float* l, float* h) {
              unsigned long long* p = a.rec + 3 * static_cast<size_t>(c);
              unsigned long long w0 = 0, w1 = 0, w2 = 0;
              const bool ok = AwaitTagged(p, a.wait_tag, a.spin_limit, &w0) &&
                              AwaitTagged(p + 1, a.wait_tag, a.spin_limit, &w1) &&
                              AwaitTagged(p + 2, a.wait_tag, a.spin_limit, &w2);
              *m = __uint_as_float(static_cast<uint32_t>(w0));
              *l = __uint_as_float(static_cast<uint32_t>(w1));
              *h = __uint_as_float(static_cast<uint32_t>(w2));
              return ok;
            },
            [&](int i, int page) {
              out[i] = page;
              PutTagged(sel + i, a.epoch, static_cast<uint32_t>(page));
            },
            emit_count, a.queries + static_cast<size_t>(r) * pool.elements, pool.summaries,
            pool.token_counts, pool.capacity, a.cand_ids + begin, pool.elements, a.scale,
            a.exact_pages, SelectAssist{}, nullptr, a.fail);
      }
      if (a.stamps != nullptr && threadIdx.x == 0) sh.stamp[2] = wall_clock64();
    }
  } else {
    const int r = item_r;
    const int head = item_sub;
    unsigned long long* sel = w.sel_rec + static_cast<size_t>(r) * stride;
    // Each thread reads its id word along with thread 0's read of the count:
    // when the select finished before this item started (most items), the
    // ids arrive in the same round trip; a word not yet current is polled
    // below.
    const unsigned long long early =
        static_cast<int>(threadIdx.x) < stride ? LoadWord(sel + threadIdx.x) : 0ull;
    if (threadIdx.x == 0) {
      unsigned long long word = 0;
      int count = 0;
      if (AwaitTagged(w.cnt_rec + r, a.wait_tag, a.spin_limit, &word)) {
        count = static_cast<int>(static_cast<uint32_t>(word));
      } else {
        ReportFailure(a.fail, kFailWait);
      }
      sh.count = count < stride ? count : stride;
    }
    __syncthreads();
    const int count = sh.count;
    for (int i = threadIdx.x; i < count; i += kFThreads) {
      unsigned long long word = i == static_cast<int>(threadIdx.x) ? early : 0ull;
      int page = -1;  // never attended (InPool fails)
      if (static_cast<unsigned>(word >> 32) == a.wait_tag ||
          AwaitTagged(sel + i, a.wait_tag, a.spin_limit, &word)) {
        page = static_cast<int>(static_cast<uint32_t>(word));
      } else {
        ReportFailure(a.fail, kFailWait);
      }
      sh.page[i] = page;
    }
    __syncthreads();
    AttentionArgs args;
    args.queries = a.queries;
    args.scale = a.scale;
    args.outputs = a.outputs;
    AttentionFastHead<128, kWideAttnLpt, kWideAttnWaves, kWideAttnUnroll>(
        pool, args, head, r, threadIdx.x, sh.page, count, sh.attn);
  }
  if (a.stamps != nullptr && threadIdx.x == 0) {
    unsigned long long* st = a.stamps + static_cast<size_t>(kWideStamps) * item;
    st[0] = sh.stamp[0];
    st[1] = static_cast<unsigned long long>(kind) | (static_cast<unsigned long long>(item_r) << 8) |
            (static_cast<unsigned long long>(blockIdx.x) << 32);
    st[2] = sh.stamp[1];
    st[3] = sh.stamp[2];
    st[4] = wall_clock64();
  }
}

// One thread advances a captured wide step's epoch (as EpochBumpKernel:
// within [2^30, 2^31)) and its launch count (the parity picks the counter
// set).
__global__ void WideBumpKernel(unsigned* epoch, unsigned* seq) {
  if (threadIdx.x == 0) {
    *epoch = ((*epoch + 1u) & 0x3FFFFFFFu) | 0x40000000u;
    *seq = *seq + 1u;
  }
}

__global__ __launch_bounds__(kFThreads) void WideStepKernel(PoolView pool, WideArgs w) {
  __shared__ WideShared sh;
  if (w.a.epoch_src != nullptr) {
    // Replayed from a captured graph: the epoch and the counter set that
    // the bump kernel just before this launch advanced.
    w.a.epoch = *w.a.epoch_src;
    w.a.wait_tag = w.a.epoch | w.a.wait_mask;
    w.a.fail.epoch = w.a.epoch;
    const unsigned n = *w.seq_src;
    w.counters = w.capture_counters + (n & 1u) * static_cast<size_t>(w.counter_words);
    w.next_counters = w.capture_counters + ((n + 1u) & 1u) * static_cast<size_t>(w.counter_words);
  }
  if (blockIdx.x == 0) {
    // Zero the other counter set for the next launch (the launch before
    // this one used it and has finished).
    for (int t = static_cast<int>(threadIdx.x); t < w.counter_words; t += kFThreads) {
      __hip_atomic_store(w.next_counters + t, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  int item = static_cast<int>(blockIdx.x);
  if (w.tickets) {
    if (threadIdx.x == 0) {
      // A spare workgroup that starts after every item was taken sees so
      // with a load and leaves without touching the counter.
      unsigned t = static_cast<unsigned>(w.items);
      if (__hip_atomic_load(w.counters, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) <
          static_cast<unsigned>(w.items)) {
        t = __hip_atomic_fetch_add(w.counters, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      sh.item = t < static_cast<unsigned>(w.items) ? static_cast<int>(t) : w.items;
    }
    __syncthreads();
    item = sh.item;
  }
  if (item < w.items) WideStepItem(pool, w, item, sh);
}

}  // namespace

void LaunchScoreExact(const PoolView& pool, const float* d_queries,
                      const int* d_cand_offsets, const int* d_cand_ids,
                      int batch, int total_candidates, int max_candidates, float scale,
                      float* d_scores, FailReport fail, hipStream_t stream,
                      const int* d_undecided) {
  if (batch <= 0 || max_candidates <= 0) return;
  // The chains kernel up to a round of its workgroups (two per CU); beyond it
  // runs several, and a lane per page then fills the chip as well (E = 1024:
  // 16000 pages 20.8 us and 25.0 with lanes, 30000 38.2 and 28.8, 60000 92 and
  // 50; E = 512: 12.3 and 14.1, 22.0 and 16.8, 39.9 and 23.3).  Requests left
  // undecided are few of the batch: always chains.
  const bool chains = pool.elements % kWave == 0 &&
                      (d_undecided != nullptr || total_candidates <= 512 * kChainPages);
  if (!chains && d_undecided != nullptr) {
    throw std::invalid_argument("undecided requests need E % 64 == 0");
  }
  if (chains) {
    // The fewest pages per workgroup that keep the batch within that round.
    int pages = kChainPages / 4;
    while (pages < kChainPages && total_candidates > 512 * pages) pages *= 2;
    hipLaunchKernelGGL(ScoreChainsKernel, dim3((max_candidates + pages - 1) / pages, batch),
                       dim3(kChainThreads), 0, stream, d_queries, pool.summaries,
                       pool.token_counts, pool.capacity, d_cand_offsets, d_cand_ids,
                       total_candidates, pages, pool.elements, scale, d_scores, d_undecided, fail);
    DSD_HIP_CHECK(hipGetLastError());
    return;
  }
  const dim3 grid((max_candidates + kWave - 1) / kWave, batch);
  if (pool.elements % 4 == 0) {
    hipLaunchKernelGGL(ScoreExactKernel<true>, grid, dim3(kWave), 0, stream,
                       d_queries, pool.summaries, pool.token_counts, pool.capacity,
                       d_cand_offsets, d_cand_ids, total_candidates, pool.elements, scale,
                       d_scores, fail);
  } else {
    hipLaunchKernelGGL(ScoreExactKernel<false>, grid, dim3(kWave), 0, stream,
                       d_queries, pool.summaries, pool.token_counts, pool.capacity,
                       d_cand_offsets, d_cand_ids, total_candidates, pool.elements, scale,
                       d_scores, fail);
  }
  DSD_HIP_CHECK(hipGetLastError());
}

bool CertifiedScoringSupported(int elements, int max_candidates, int top_k) {
  if (elements % kWave != 0 || elements < kWave) return false;
  if (max_candidates <= kCertMaxKeys) return true;
  return max_candidates <= kLargeMaxKeys && top_k <= kLargeMaxK;
}

bool CertifiedSelectMayDefer(int max_candidates) { return max_candidates > kCertMaxKeys; }

void LaunchScoreBounds(const PoolView& pool, const float* d_queries,
                       const int* d_cand_offsets, const int* d_cand_ids, int batch,
                       int total_candidates, int max_candidates, float scale, float* d_mid,
                       float* d_lo, float* d_hi, FailReport fail, hipStream_t stream) {
  if (batch <= 0 || max_candidates <= 0) return;
  if (pool.elements == 4096) {
    // The fused step's float score passes, 8..128 pages per workgroup.
    LaunchScorePages(pool, d_queries, d_cand_offsets, d_cand_ids, batch, total_candidates,
                     max_candidates, scale, d_mid, d_lo, d_hi, fail, stream);
    return;
  }
  // More waves than the chip holds at once (7168), so that one that ends makes
  // room: a page per wave up to 16384 pages (32 requests of 8 x 128 heads and
  // 300 pages each, with the present select: the step 42.9 us, 44.8 with 8192
  // waves, 47.0 with 4096).  Beyond E = 4096 a workgroup's copy of the query
  // weighs more, and up to 8192 pages a wave takes two (16 requests of 500 pages,
  // 40, 64 and 80 heads of 128: 52.2, 84.0 and 112.2 us; 54.3, 85.7 and 112.4 with
  // one; 32 of 300 pages, one a wave: 76.1, 108.3 and 143.9 us; 81.6, 116.2 and
  // 153.2 with three).
  const int target_waves = pool.elements > 4096 && total_candidates <= 8192 ? 4096 : 16384;
  const int per_wave = std::min(
      kWave, std::max(1, (total_candidates + target_waves - 1) / target_waves));
  const int per_group = per_wave * kBoundWaves;
  const dim3 grid((max_candidates + per_group - 1) / per_group, batch);
  const dim3 block(kBoundWaves * kWave);
  const size_t query_bytes = sizeof(float) * static_cast<size_t>(pool.elements);
  if (pool.elements <= 4 * kWave) {
    hipLaunchKernelGGL((ScoreBoundGenericKernel<false, 1>), grid, block, 0, stream, d_queries,
                       pool.summaries, pool.token_counts, pool.capacity, d_cand_offsets,
                       d_cand_ids, total_candidates, per_wave, pool.elements, scale, d_mid, d_lo,
                       d_hi, fail);
  } else if (query_bytes <= kBoundQueryLds) {
    hipLaunchKernelGGL((ScoreBoundGenericKernel<true, kBoundRows>), grid, block, query_bytes,
                       stream, d_queries, pool.summaries, pool.token_counts, pool.capacity,
                       d_cand_offsets, d_cand_ids, total_candidates, per_wave, pool.elements,
                       scale, d_mid, d_lo, d_hi, fail);
  } else {
    hipLaunchKernelGGL((ScoreBoundGenericKernel<false, kBoundRows>), grid, block, 0, stream,
                       d_queries, pool.summaries, pool.token_counts, pool.capacity,
                       d_cand_offsets, d_cand_ids, total_candidates, per_wave, pool.elements,
                       scale, d_mid, d_lo, d_hi, fail);
  }
  DSD_HIP_CHECK(hipGetLastError());
}

void LaunchSelectCertified(const PoolView& pool, const float* d_mid, const float* d_lo,
                           const float* d_hi,
                           const float* d_queries,
                           const int* d_cand_offsets, const int* d_cand_ids, int batch,
                           int total_candidates, int max_candidates, float scale, int top_k,
                           int* d_selected, int* d_counts, int* d_exact_pages, FailReport fail,
                           hipStream_t stream, const SelectAssist& assist) {
  if (batch <= 0) return;
  if (max_candidates <= kRankMax) {
    // Always four waves: three of them form products while wave 0 runs the
    // exact chains.
    hipLaunchKernelGGL(SelectCertifiedRankKernel, dim3(batch), dim3(kRankMax), 0, stream,
                       d_mid, d_lo, d_hi, d_queries, pool.summaries, pool.token_counts,
                       pool.capacity, d_cand_offsets, d_cand_ids, total_candidates,
                       max_candidates, pool.elements, scale, top_k, d_selected, d_counts,
                       d_exact_pages, fail);
    DSD_HIP_CHECK(hipGetLastError());
    return;
  }
  if (pool.elements % kWave != 0) {
    throw std::invalid_argument("certified select needs E % 64 == 0");
  }
  if (max_candidates > kCertMaxKeys && (max_candidates > kLargeMaxKeys || top_k > kLargeMaxK)) {
    throw std::invalid_argument("certified select supports up to " +
                                std::to_string(kLargeMaxKeys) + " candidates per request and " +
                                std::to_string(kLargeMaxK) + " of them selected");
  }
  const auto kernel = max_candidates <= kCertMaxKeys
                          ? SelectCertifiedKernel<kCertMaxKeys / kSelThreads, CertShared>
                      : max_candidates <= kLargeMaxKeys / 2
                          ? SelectCertifiedKernel<kLargeMaxKeys / 2 / kSelThreads, CertSharedLarge>
                          : SelectCertifiedKernel<kLargeMaxKeys / kSelThreads, CertSharedLarge>;
  // Helpers only where every workgroup is resident at once, so that a
  // request's workgroup and its helpers do run side by side (one that does
  // not run in time costs the bounded wait, nothing else).
  SelectAssist a = assist;
  a.helpers = a.words == nullptr || a.epoch == 0
                  ? 0
                  : std::min(kAssistMaxHelpers, a.compute_units / batch - 1);
  if (a.helpers < kAssistLeastPages) a.helpers = 0;
  hipLaunchKernelGGL(kernel, dim3(batch * (1 + a.helpers)), dim3(kSelThreads), 0, stream, d_mid,
                     d_lo, d_hi, d_queries, pool.summaries, pool.token_counts, pool.capacity,
                     d_cand_offsets, d_cand_ids, batch, total_candidates, max_candidates,
                     pool.elements, scale, top_k, d_selected, d_counts, d_exact_pages, a, fail);
  DSD_HIP_CHECK(hipGetLastError());
}

int SelectMaxCandidates() { return kSelectMaxKeys; }

bool WideStepSupported(const PoolView& pool, int max_candidates, int top_k) {
  return pool.elements == kFE && pool.head_dim == 128 &&
         pool.page_size > 0 && max_candidates > 0 && max_candidates <= kCertMaxKeys &&
         top_k <= kCertMaxKeys;
}

int WideStepMaxCandidates() { return kCertMaxKeys; }

int WideStepStampsPerGroup() { return kWideStamps; }

int WideStepItems(const PoolView& pool, int batch, int groups) {
  return batch * groups + batch * pool.num_heads;
}

int WideStepGrid(int items, bool tickets) { return tickets ? items + items / 2 : items; }

void LaunchWideStep(const PoolView& pool, const WideArgs& w, hipStream_t stream) {
  if (w.a.batch <= 0) return;
  if (!WideStepSupported(pool, w.a.max_candidates, w.a.top_k)) {
    throw std::invalid_argument("the wide step needs E = 4096, head_dim 128 and at most 2048 "
                                "candidates per request");
  }
  if (w.pages_per_group <= 0 || w.pages_per_group % kFPagesPerPass != 0 ||
      static_cast<long long>(w.groups) * w.pages_per_group < w.a.max_candidates) {
    throw std::invalid_argument("wide step slices do not cover max_candidates");
  }
  if (w.a.rec == nullptr || w.sel_rec == nullptr || w.cnt_rec == nullptr ||
      w.counters == nullptr || w.next_counters == nullptr || w.counter_words < w.a.batch + 1 ||
      w.a.sel_stride < (w.a.top_k > 0 ? w.a.top_k : 1)) {
    throw std::invalid_argument("wide step scratch missing");
  }
  if (w.a.epoch_src != nullptr) {
    if (w.seq_src == nullptr || w.capture_counters == nullptr) {
      throw std::invalid_argument("a captured wide step needs its device launch count");
    }
    hipLaunchKernelGGL(WideBumpKernel, dim3(1), dim3(kWave), 0, stream,
                       const_cast<unsigned*>(w.a.epoch_src), w.seq_src);
    DSD_HIP_CHECK(hipGetLastError());
  }
  if (w.items != WideStepItems(pool, w.a.batch, w.groups)) {
    throw std::invalid_argument("wide step item count does not match its slices");
  }
  const int grid = WideStepGrid(w.items, w.tickets);
  hipLaunchKernelGGL(WideStepKernel, dim3(grid), dim3(kFThreads), 0, stream, pool, w);
  DSD_HIP_CHECK(hipGetLastError());
}

void LaunchSelectTopK(const float* d_scores, const int* d_cand_offsets,
                      const int* d_cand_ids, int batch, int total_candidates,
                      int max_candidates, int top_k, int* d_selected, int* d_counts,
                      FailReport fail, hipStream_t stream, bool undecided_only) {
  if (batch <= 0) return;
  int m = 1;
  while (m < max_candidates) m <<= 1;
  if (m > kSelectMaxKeys) {
    throw std::invalid_argument(
        "candidate pages per request exceed the top-k select limit of " +
        std::to_string(kSelectMaxKeys));
  }
  int threads = m / 2;
  if (threads < kWave) threads = kWave;
  if (threads > 256) threads = 256;
  hipLaunchKernelGGL(SelectTopKKernel, dim3(batch), dim3(threads),
                     sizeof(uint64_t) * static_cast<size_t>(m), stream, d_scores,
                     d_cand_offsets, d_cand_ids, total_candidates, max_candidates, top_k,
                     d_selected, d_counts, undecided_only, fail);
  DSD_HIP_CHECK(hipGetLastError());
}

void PreloadStepKernels() {
  PreloadKernel(WideStepKernel);
  PreloadKernel(WideBumpKernel);
  PreloadKernel(SelectCertifiedKernel<kCertMaxKeys / kSelThreads, CertShared>);
  PreloadKernel(SelectCertifiedKernel<kLargeMaxKeys / 2 / kSelThreads, CertSharedLarge>);
  PreloadKernel(SelectCertifiedKernel<kLargeMaxKeys / kSelThreads, CertSharedLarge>);
  PreloadKernel(SelectCertifiedRankKernel);
  PreloadKernel(SelectTopKKernel);
  PreloadKernel(ScoreBoundGenericKernel<true, kBoundRows>);
  PreloadKernel(ScoreBoundGenericKernel<false, 1>);
  PreloadKernel(ScoreChainsKernel);
}

}  // namespace dsdk
