// attention.hip -- fused gather + softmax attention over page lists (gfx950):
// the three-kernel step's last stage (reference GatherPagesCpu +
// SparseAttentionCpu, src/reference_kernels.cpp:109-194) and dense attention
// (DenseAttentionCpu, :196-203), whose list is every candidate page.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>

#include "attention_head.h"
#include "dsd_internal.h"
#include "score_slice.h"
#include "step_common.h"

namespace dsdk {
namespace {

// ---------------------------------------------------------------------------
// Any head_dim <= 256 (flash-decoding inside a workgroup).
//
// Workgroup = (head h, request r); its waves stride over 16-token chunks of
// the request's page list.  Lane (g, j) = (lane/4, lane%4) owns token slot g
// of the chunk and the j-th quarter of the head's dims, so a 4-lane group
// reads one 4*DQ-float K row and one V row (contiguous, vectorised).  Each
// lane keeps its own online-softmax stream (m, l, acc[DQ]) over the tokens
// it sees: the only per-token cross-lane traffic is the 2-step dot-product
// reduction within the group.  Streams are merged once at the end: across
// the 16 token slots with xor shuffles, across waves through LDS.  Logits
// live in the log2 domain (q pre-scaled by scale*log2 e) so each exponential
// is one v_exp_f32.
// ---------------------------------------------------------------------------
constexpr int kAttnWaves = 4;
constexpr int kAttnThreads = kAttnWaves * kWave;
constexpr int kChunk = 16;
// DQ > 0: head_dim == 4*DQ, lane j covers dims [j*DQ, (j+1)*DQ).
// DQ == 0: generic head_dim <= 256, lane j covers dims j, j+4, j+8, ...
template <int DQ>
__global__ __launch_bounds__(kAttnThreads) void AttentionKernel(
    PoolView pool, AttentionArgs args) {
  constexpr int kRegs = DQ > 0 ? DQ : 64;
  const int h = blockIdx.x;
  const int r = blockIdx.y;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  const int g = lane >> 2;
  const int j = lane & 3;
  const int D = pool.head_dim;
  const int E = pool.elements;
  const int ps = pool.page_size;

  int start, count;
  if (args.list_stride > 0) {
    start = r * args.list_stride;
    count = args.list_counts[r];
  } else {
    start = args.list_offsets[r];
    count = args.list_offsets[r + 1] - start;
  }

  const int nd = DQ > 0 ? DQ : (D - j + 3) / 4;
  const int dim0 = DQ > 0 ? j * DQ : j;
  const int dstep = DQ > 0 ? 1 : 4;
  const int head_off = h * D + dim0;

  float q[kRegs];
  float acc[kRegs];
  {
    const float qscale = args.scale * kLog2e;
    const float* qp = args.queries + static_cast<size_t>(r) * E + head_off;
    if constexpr (DQ > 0) {
      LoadDims<DQ>(qp, q);
    } else {
#pragma unroll
      for (int i = 0; i < kRegs; ++i) q[i] = i < nd ? qp[i * dstep] : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < kRegs; ++i) {
      q[i] *= qscale;
      acc[i] = 0.0f;
    }
  }

  float m = -INFINITY;
  float l = 0.0f;
  const int total = count * ps;
  for (int base = wave * kChunk; base < total; base += kAttnWaves * kChunk) {
    const int f = base + g;
    bool valid = false;
    float kv[kRegs];
    float vv[kRegs];
    if (f < total) {
      const int slot = f / ps;
      const int t = f - slot * ps;
      const int page = args.list_ids[start + slot];
      valid = InPool(page, pool.capacity) && t < pool.token_counts[page];
      if (valid) {
        const size_t off = static_cast<size_t>(page) * pool.page_elems +
                           static_cast<size_t>(t) * E + head_off;
        if constexpr (DQ > 0) {
          LoadDims<DQ>(pool.keys + off, kv);
          LoadDims<DQ>(pool.values + off, vv);
        } else {
#pragma unroll
          for (int i = 0; i < kRegs; ++i) {
            kv[i] = i < nd ? pool.keys[off + i * dstep] : 0.0f;
            vv[i] = i < nd ? pool.values[off + i * dstep] : 0.0f;
          }
        }
      }
    }
    float dot = 0.0f;
    if (valid) {
#pragma unroll
      for (int i = 0; i < kRegs; ++i) dot = fmaf(q[i], kv[i], dot);
    }
    dot += __shfl_xor(dot, 1, kWave);
    dot += __shfl_xor(dot, 2, kWave);
    if (valid) {
      const float m_new = fmaxf(m, dot);
      const float alpha = Exp2(m - m_new);
      const float beta = Exp2(dot - m_new);
      l = fmaf(l, alpha, beta);
#pragma unroll
      for (int i = 0; i < kRegs; ++i) acc[i] = fmaf(acc[i], alpha, beta * vv[i]);
      m = m_new;
    }
  }

  // Merge the 16 token-slot streams of this wave (lanes differing in g).
  float wm = m;
#pragma unroll
  for (int o = 4; o < kWave; o <<= 1) wm = fmaxf(wm, __shfl_xor(wm, o, kWave));
  const float sc = (m == -INFINITY) ? 0.0f : Exp2(m - wm);
  float wl = l * sc;
#pragma unroll
  for (int i = 0; i < kRegs; ++i) acc[i] *= sc;
#pragma unroll
  for (int o = 4; o < kWave; o <<= 1) {
    wl += __shfl_xor(wl, o, kWave);
#pragma unroll
    for (int i = 0; i < kRegs; ++i) acc[i] += __shfl_xor(acc[i], o, kWave);
  }

  // Merge the waves through LDS: s_acc[wave][D], s_m/s_l[wave].
  extern __shared__ float smem[];
  float* s_m = smem;
  float* s_l = smem + kAttnWaves;
  float* s_acc = smem + 2 * kAttnWaves;
  if (g == 0) {
    if (j == 0) {
      s_m[wave] = wm;
      s_l[wave] = wl;
    }
#pragma unroll
    for (int i = 0; i < kRegs; ++i) {
      if (i < nd) s_acc[wave * D + dim0 + i * dstep] = acc[i];
    }
  }
  __syncthreads();
  float mx = -INFINITY;
#pragma unroll
  for (int w = 0; w < kAttnWaves; ++w) mx = fmaxf(mx, s_m[w]);
  float* out = args.outputs + static_cast<size_t>(r) * E + static_cast<size_t>(h) * D;
  for (int d = threadIdx.x; d < D; d += kAttnThreads) {
    float lt = 0.0f;
    float at = 0.0f;
    if (mx != -INFINITY) {
#pragma unroll
      for (int w = 0; w < kAttnWaves; ++w) {
        const float s = (s_m[w] == -INFINITY) ? 0.0f : Exp2(s_m[w] - mx);
        lt = fmaf(s_l[w], s, lt);
        at = fmaf(s_acc[w * D + d], s, at);
      }
    }
    // No valid token at all: the reference returns zeros
    // (src/cuda/sparse_batched_attention.cu:364-369; CPU :159-161).
    out[d] = lt == 0.0f ? 0.0f : at / lt;
  }
}

// ---------------------------------------------------------------------------
// The head sizes with a float4 lane split (attention_head.h), optionally with
// a head's tokens spread over several workgroups.
//
// Bound by HBM: each K and V row is read once (0.5 flop per byte).
//
// Unsplit (kSplit false, piece_room 0): workgroup (h, r) attends request r's
// whole list.  A kernel of its own: beside the pieces' code the compiler gives
// the token loop a schedule that is 1-5% slower.
// A batch of few requests then runs few workgroups: one request of 32 heads
// and 32768 tokens kept 32 of 256 CUs busy (dense, 1.07 GB: 1234 us).
//
// Split: grid (heads, batch + room).  The batch's token slots are cut into
// pieces of P slots, P = the total over `room`, so that request r gets
// max(1, ceil(slots_r / P)) pieces, at most batch + room in all; workgroup
// (h, g) finds piece g by a scan of the lists' lengths (the lengths are
// device data, so the host cannot).  Pieces are equal whatever the lengths:
// a ragged batch has no long tail.  A request of one piece writes its output;
// the others publish (m, l, acc) as tagged words, and the workgroup that
// arrives last at the request's counter merges them in piece order (the
// result does not depend on which workgroup that is) and zeroes the words and
// the counter for the next launch on the same scratch.  The words carry the
// launch's tag, so nothing orders them but the tag (no fence, which would write
// back the XCD's L2).  Every wait ends: the merging workgroup waits only for
// words whose stores were issued before their workgroup arrived; the poll is
// bounded anyway, a word that never came is reported (kFailWait, zero outputs;
// NaN from a dense step, which reports nothing) and not taken for a later
// launch's.  The request above takes 185 us (5.8 TB/s).
//
// Either way the list's ids and token counts are staged in LDS, 256 entries
// at a time, instead of a chain of two loads ahead of every chunk's rows
// (dense, 16 requests of 512-2048 tokens: 118 us against 125).
// ---------------------------------------------------------------------------
constexpr int kAttnTile = 256;       // list entries per LDS tile
constexpr int kAttnMaxPieces = 256;  // per request (room), the merge's LDS
// Workgroups of 8 waves the chip runs at once (two per CU).
constexpr int kAttnRound = 512;
constexpr int kAttnWhole = 3;

// Token slots of request b (a malformed, negative or overflowing length holds none).
__device__ __forceinline__ int ListSlots(const AttentionArgs& a, int b, int ps, int* start) {
  int count;
  if (a.list_stride > 0) {
    *start = b * a.list_stride;
    count = a.list_counts[b];
  } else {
    *start = a.list_offsets[b];
    count = a.list_offsets[b + 1] - *start;
  }
  return count > 0 ? max(count * ps, 0) : 0;
}

struct AttnPiece {
  int r = 0;       // request
  int start = 0;   // its list
  int index = 0;   // this piece of
  int pieces = 1;  // its pieces
  int f0 = 0;      // token slots [f0, f1)
  int f1 = 0;
};

// x of the DPP source lane (step_common.h), 0 where there is none.
template <int kCtrl, int kRowMask = 0xf>
__device__ __forceinline__ int DppMoveI(int x) {
  return __builtin_amdgcn_update_dpp(0, x, kCtrl, kRowMask, 0xf, true);
}

__device__ __forceinline__ int WaveInclusiveScanI(int x) {
  x += DppMoveI<kRowShr1>(x);
  x += DppMoveI<kRowShr2>(x);
  x += DppMoveI<kRowShr4>(x);
  x += DppMoveI<kRowShr8>(x);
  x += DppMoveI<kRowBcast15, 0xa>(x);
  x += DppMoveI<kRowBcast31, 0xc>(x);
  return x;
}

// The largest of the lanes' x >= 0, in every lane.
__device__ __forceinline__ int WaveMaxI(int x) {
  x = max(x, DppMoveI<kRowShr1>(x));
  x = max(x, DppMoveI<kRowShr2>(x));
  x = max(x, DppMoveI<kRowShr4>(x));
  x = max(x, DppMoveI<kRowShr8>(x));
  x = max(x, DppMoveI<kRowBcast15, 0xa>(x));
  x = max(x, DppMoveI<kRowBcast31, 0xc>(x));
  return __builtin_amdgcn_readlane(x, kWave - 1);
}

// Piece g of the batch, pieces of a multiple of kAlign slots; false beyond
// the last one.  Every wave computes the same.
//
// Whether to split at all.  The longest request is the launch's tail only where
// it has more slots than its share of the chip's time, the mean times
// piece_share * batch (PieceShare), and splitting costs a merge (7-11 us of a
// head's stream: kAttnWhole steps, 384 slots at least).  Measured, split and
// whole, 128 dims: 4 x 32 equal heads of 600 slots 20.5 and 18.8 us, of 1500
// 35.6 and 39.8; 8 x 32 of 1500 72.3 and 67.1, of 375-1500 44.8 and 45.6, of
// 1250-5000 164 and 174; 15 x 32 of 600 57.2 and 50.3; 60 x 4 of 256 dims, 600
// slots, 57.2 and 45.4.  A request of at most kAttnWhole steps is one piece
// (one of 32 heads: 300 tokens 11.0 us in three pieces and 10.4 in one).
template <int kAlign>
__device__ __forceinline__ bool FindPiece(const AttentionArgs& a, int ps, int g, AttnPiece* out) {
  constexpr int kGain = kAttnWhole * kAlign > 384 ? kAttnWhole * kAlign : 384;
  const int lane = threadIdx.x & (kWave - 1);
  double total = 0.0;  // (exact: below 2^53)
  int longest = 0;
  int start0 = 0, slots0 = 0;  // requests 0..63 (loaded once)
  for (int b = lane; b < a.batch; b += kWave) {
    int start;
    const int slots = ListSlots(a, b, ps, &start);
    if (b < kWave) {
      start0 = start;
      slots0 = slots;
    }
    total += static_cast<double>(slots);
    longest = max(longest, slots);
  }
  total = ReadLaneD(WaveInclusiveScanD(total), kWave - 1);
  longest = WaveMaxI(longest);
  if (static_cast<double>(longest - kGain) <= total * static_cast<double>(a.piece_share)) {
    if (g >= a.batch) return false;
    out->r = g;
    if (g < kWave) {
      out->start = __builtin_amdgcn_readlane(start0, g);
      out->f1 = __builtin_amdgcn_readlane(slots0, g);
    } else {
      out->f1 = ListSlots(a, g, ps, &out->start);
    }
    return true;
  }
  const double share = ceil(total / static_cast<double>(a.piece_room));
  const int P = share >= 0x1p30
                    ? 0x40000000
                    : max(1, (static_cast<int>(share) + kAlign - 1) / kAlign) * kAlign;
  int before = 0;
  for (int b0 = 0; b0 < a.batch; b0 += kWave) {
    const int b = b0 + lane;
    int start = start0, slots = slots0;
    if (b0 > 0) slots = b < a.batch ? ListSlots(a, b, ps, &start) : 0;
    int n = b < a.batch ? 1 : 0;
    if (slots > kAttnWhole * kAlign) n = (slots - 1) / P + 1;
    const int incl = WaveInclusiveScanI(n);
    const int first = before + incl - n;
    const uint64_t mine = __ballot(g >= first && g < first + n);
    if (mine != 0) {
      const int l = __ffsll(static_cast<long long>(mine)) - 1;
      out->r = b0 + l;
      out->start = __builtin_amdgcn_readlane(start, l);
      out->pieces = __builtin_amdgcn_readlane(n, l);
      out->index = g - __builtin_amdgcn_readlane(first, l);
      const int all = __builtin_amdgcn_readlane(slots, l);
      out->f0 = out->index * P;
      out->f1 = out->pieces == 1 || all - out->f0 < P ? all : out->f0 + P;
      return true;
    }
    before += __builtin_amdgcn_readlane(incl, kWave - 1);
  }
  return false;
}

// A published word's value once it carries the launch's tag, zeroed for the
// next launch; *late when it never did (the word stays: the next launch has
// another tag).
__device__ __forceinline__ float TakeWord(const AttentionArgs& args, unsigned long long* p,
                                          int* late) {
  const unsigned tag = args.piece_tag | args.piece_wait_mask;
  unsigned long long w = LoadWord(p);
  for (unsigned i = 0; static_cast<unsigned>(w >> 32) != tag; ++i) {
    if (i >= args.piece_spin_limit || *static_cast<volatile int*>(late) != 0) {
      *late = 1;
      return 0.0f;
    }
    __builtin_amdgcn_s_sleep(1);
    w = LoadWord(p);
  }
  __hip_atomic_store(p, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return __uint_as_float(static_cast<uint32_t>(w));
}

// A split head's piece p (its waves' merged state in thread tid < D): published,
// and all of the head's merged by the last workgroup to arrive.
template <int D, int WAVES>
__device__ __forceinline__ void MergePieces(const PoolView& pool, const AttentionArgs& args,
                                            const AttnPiece& p, int h, float mx, float lt,
                                            float at, AttnFastShared<WAVES, D>& sh, float* out) {
  constexpr int kThreads = WAVES * kWave;
  __shared__ float s_pm[kAttnMaxPieces];
  __shared__ float s_pl[kAttnMaxPieces];
  __shared__ int s_last;
  __shared__ int s_late;
  const int tid = threadIdx.x;
  unsigned long long* words =
      args.piece_words +
      (static_cast<size_t>(blockIdx.y) * pool.num_heads + h) * static_cast<size_t>(D + 2);
  if (tid < D) {
    if (tid == 0) {
      PutTagged(words, args.piece_tag, __float_as_uint(mx));
      PutTagged(words + 1, args.piece_tag, __float_as_uint(lt));
    }
    PutTagged(words + 2 + tid, args.piece_tag, __float_as_uint(at));
  }
  __syncthreads();
  unsigned* arrivals = args.piece_arrivals + static_cast<size_t>(p.r) * pool.num_heads + h;
  if (tid == 0) {
    const unsigned prev =
        __hip_atomic_fetch_add(arrivals, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = prev == static_cast<unsigned>(p.pieces - 1) ? 1 : 0;
    s_late = 0;
  }
  __syncthreads();
  if (s_last == 0) return;
  if (tid == 0) {
    __hip_atomic_store(arrivals, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  // The request's pieces are consecutive: words of piece i of them.
  const size_t stride = static_cast<size_t>(pool.num_heads) * (D + 2);
  unsigned long long* first = words - static_cast<size_t>(p.index) * stride;
  for (int i = tid; i < p.pieces; i += kThreads) {
    s_pm[i] = TakeWord(args, first + i * stride, &s_late);
    s_pl[i] = TakeWord(args, first + i * stride + 1, &s_late);
  }
  __syncthreads();
  float m = kNoMax;
  for (int i = 0; i < p.pieces; ++i) m = fmaxf(m, s_pm[i]);
  constexpr int kGroups = kThreads / D;  // piece i by thread group i mod kGroups
  const int d = tid % D;
  const int grp = tid / D;
  lt = 0.0f;
  at = 0.0f;
  if (grp < kGroups) {
    for (int i = grp; i < p.pieces; i += kGroups) {
      const float a = TakeWord(args, first + i * stride + 2 + d, &s_late);
      const float sw = Exp2(s_pm[i] - m);
      lt = fmaf(s_pl[i], sw, lt);
      at = fmaf(a, sw, at);
    }
  }
  // (sh.m / sh.l / sh.acc were last read before the arrival's barriers)
  static_assert(kGroups <= WAVES, "a group per wave slot of the shared states");
  if (grp < kGroups) {
    sh.acc[grp][d] = at;
    if (d == 0) sh.l[grp] = lt;
  }
  __syncthreads();
  if (tid < D) {
    lt = 0.0f;
    at = 0.0f;
    for (int i = 0; i < kGroups; ++i) {
      lt += sh.l[i];
      at += sh.acc[i][tid];
    }
    float o = AttnOutput(m, lt, at);
    if (s_late != 0) {
      // Zeros and a report, as the step's other waits; NaN where the launch
      // has nowhere to report to.
      if (tid == 0) ReportFailure(args.fail, kFailWait);
      o = args.fail.word != nullptr ? 0.0f : NAN;
    }
    out[tid] = o;
  }
}

template <int D, int LPT, int WAVES, int UNROLL, bool kSplit>
__global__ __launch_bounds__(WAVES * kWave) void AttentionFastKernel(
    PoolView pool, AttentionArgs args) {
  constexpr int DQ = D / LPT;
  constexpr int kThreads = WAVES * kWave;
  constexpr int kAlign = WAVES * (kWave / LPT) * UNROLL;
  static_assert(kThreads >= D, "a thread per dim");
  __shared__ AttnFastShared<WAVES, D> sh;
  __shared__ int s_page[kAttnTile];
  __shared__ int s_ntok[kAttnTile];
  const int h = blockIdx.x;
  const int tid = threadIdx.x;
  const int ps = pool.page_size;
  AttnPiece p;
  if constexpr (!kSplit) {
    p.r = blockIdx.y;
    p.f1 = ListSlots(args, p.r, ps, &p.start);
  } else if (!FindPiece<kAlign>(args, ps, blockIdx.y, &p)) {
    return;
  }
  const int head_off = h * D + (tid & (kWave - 1)) % LPT * DQ;
  AttnState<DQ> st;
  AttnBegin<DQ>(args.queries + static_cast<size_t>(p.r) * pool.elements + head_off, args.scale,
                st);
  // Tiles of list entries: ids and token counts in LDS, so that a chunk's
  // rows load without a chain of two loads before them.  (256 entries are a
  // whole number of steps whatever the page size, so an unsplit head's waves
  // see the slots they would see without tiles.)
  const int s_end = (p.f1 + ps - 1) / ps;
  for (int s0 = p.f0 / ps; s0 < s_end; s0 += kAttnTile) {
    const int n = s_end - s0 < kAttnTile ? s_end - s0 : kAttnTile;
    if (s0 * ps > p.f0) __syncthreads();  // the previous tile has been read
    for (int i = tid; i < n; i += kThreads) {
      const int page = args.list_ids[p.start + s0 + i];
      s_page[i] = page;
      s_ntok[i] = InPool(page, pool.capacity) ? pool.token_counts[page] : 0;
    }
    __syncthreads();
    const int f0 = s0 * ps > p.f0 ? s0 * ps : p.f0;
    const int f1 = n < kAttnTile || (s0 + n) * ps > p.f1 ? p.f1 : (s0 + n) * ps;
    AttnRange<D, LPT, WAVES, UNROLL, kSplit>(
        pool, head_off, tid, f0, f1,
        [&](int s, int t, int* page) {
          *page = s_page[s - s0];
          return t < s_ntok[s - s0];
        },
        st);
  }
  AttnMergeWave<D, LPT, WAVES>(tid, st, sh);
  float* out = args.outputs + static_cast<size_t>(p.r) * pool.elements + static_cast<size_t>(h) * D;
  float mx = 0.0f, lt = 0.0f, at = 0.0f;
  if (tid < D) AttnCombine<D, WAVES>(sh, tid, &mx, &lt, &at);
  if (!kSplit || p.pieces == 1) {
    if (tid < D) out[tid] = AttnOutput(mx, lt, at);
    return;
  }
  if constexpr (kSplit) MergePieces<D, WAVES>(pool, args, p, h, mx, lt, at, sh, out);
}

// The share of the chip's time that a launch of `heads` equal unsplit heads
// leaves to each head's slots.  About 214 workgroups load the chip; up to 256 run
// one on a CU.  Just beyond, the CUs that got a second one are a tail of their
// own, which thins out as more do: 288 heads of 128 dims and 3000 slots take
// 150 us split and 183 whole, 352 183 and 193, 384 204 and 202, 448 229 and 225
// (64 dims: 92 and 116, 114 and 122, 125 and 126, 135 and 134).
float PieceShare(long long heads) {
  if (heads <= 214) return static_cast<float>(heads) / 214.0f;
  if (heads <= 256 || heads >= 448) return 1.0f;
  return 0.5f + 0.5f * static_cast<float>(heads - 256) / 192.0f;
}

using AttnKernelFn = void (*)(PoolView, AttentionArgs);

struct AttnVariant {
  int lpt, waves, unroll;
  AttnKernelFn fn, split;
};

#define DSD_ATTN_VARIANT(L, W, U) \
  AttnVariant{L, W, U, AttentionFastKernel<128, L, W, U, false>, \
              AttentionFastKernel<128, L, W, U, true>}
const AttnVariant kAttnVariants[] = {
    DSD_ATTN_VARIANT(4, 4, 1),  DSD_ATTN_VARIANT(4, 4, 2),  DSD_ATTN_VARIANT(4, 8, 1),
    DSD_ATTN_VARIANT(8, 4, 1),  DSD_ATTN_VARIANT(8, 4, 2),  DSD_ATTN_VARIANT(8, 4, 4),
    DSD_ATTN_VARIANT(8, 8, 1),  DSD_ATTN_VARIANT(8, 8, 2),  DSD_ATTN_VARIANT(16, 4, 2),
    DSD_ATTN_VARIANT(16, 4, 4), DSD_ATTN_VARIANT(16, 8, 2), DSD_ATTN_VARIANT(16, 8, 4),
    DSD_ATTN_VARIANT(16, 16, 4),
};
#undef DSD_ATTN_VARIANT

// The D = 128 variant in use: DSD_ATTN_VARIANT="LPTxWAVESxUNROLL" selects
// one of kAttnVariants (a tuning knob); otherwise the measured default.
const AttnVariant& SelectAttnVariant() {
  int lpt = 16, waves = 8, unroll = 4;
  if (const char* env = std::getenv("DSD_ATTN_VARIANT")) {
    int a = 0, b = 0, c = 0;
    if (std::sscanf(env, "%dx%dx%d", &a, &b, &c) == 3) {
      lpt = a;
      waves = b;
      unroll = c;
    }
  }
  for (const auto& v : kAttnVariants) {
    if (v.lpt == lpt && v.waves == waves && v.unroll == unroll) return v;
  }
  throw std::invalid_argument("unknown DSD_ATTN_VARIANT");
}

template <int DQ>
void LaunchAttentionT(const PoolView& pool, const AttentionArgs& args,
                      hipStream_t stream) {
  const size_t lds = sizeof(float) * (2 * kAttnWaves + kAttnWaves * pool.head_dim);
  hipLaunchKernelGGL(AttentionKernel<DQ>, dim3(pool.num_heads, args.batch),
                     dim3(kAttnThreads), lds, stream, pool, args);
}

// Slots per step of a head's workgroup (kAlign), 0 for the head sizes without
// a float4 lane split.
struct AttnShape {
  int waves = 0, align = 0;
  AttnKernelFn fn = nullptr, split = nullptr;  // split: null where none ever is
};

template <int D, int LPT, int WAVES, int UNROLL, bool kMaySplit = true>
AttnShape ShapeOf() {
  AttnShape shape{WAVES, WAVES * (kWave / LPT) * UNROLL,
                  AttentionFastKernel<D, LPT, WAVES, UNROLL, false>};
  if constexpr (kMaySplit) shape.split = AttentionFastKernel<D, LPT, WAVES, UNROLL, true>;
  return shape;
}

// heads: workgroups of the unsplit launch; max_slots: the lists' longest, 0:
// unknown (dense steps).  Short lists, and lists of up to 1024 slots where heads
// fill the chip, take 64 dims with one chunk in flight: half the registers, so
// more workgroups share a CU, and a short list spreads over more waves (16
// heads of 64 slots 4.6 and 5.2 us, 32 x 16 heads of 128 slots 8.8 and 9.0, of
// 512 24.2 and 25.6); with four in flight a workgroup streams longer lists
// faster where the launch waits for a few (dense, 17 x 32 heads of 500-2000
// slots 77 us, 94 with one; 20 of 200-4000 153 and 160).  80 dims: four waves for
// short lists, which wait for eight waves' merge (16 heads of 64 slots 4.5 and
// 5.1 us), eight for longer ones (16 heads of 1500 slots: 15.6 and 11.8).
AttnShape FastShape(int head_dim, bool wide, long long heads, long long max_slots) {
  if (head_dim == 128 && wide) {
    return ShapeOf<128, kWideAttnLpt, kWideAttnWaves, kWideAttnUnroll, false>();
  }
  const bool is_short = max_slots > 0 && max_slots <= (heads >= kAttnRound ? 1024 : 128);
  switch (head_dim) {
    case 64: return is_short ? ShapeOf<64, 8, 8, 1, false>() : ShapeOf<64, 8, 8, 4>();
    case 80: return is_short ? ShapeOf<80, 4, 4, 1, false>() : ShapeOf<80, 4, 8, 1>();
    case 96: return ShapeOf<96, 8, 8, 2>();
    case 128: {
      const AttnVariant& v = SelectAttnVariant();
      return AttnShape{v.waves, v.waves * (kWave / v.lpt) * v.unroll, v.fn, v.split};
    }
    case 256: return ShapeOf<256, 16, 8, 2>();
    default: return AttnShape{};
  }
}

}  // namespace

int AttentionPieceRoom(const PoolView& pool, int batch, long long max_slots) {
  const long long heads = pool.num_heads;
  const AttnShape shape = FastShape(pool.head_dim, false, batch * heads, max_slots);
  if (shape.split == nullptr || batch <= 0) return 0;
  if (max_slots > 0 && max_slots <= kAttnWhole * shape.align) return 0;  // one piece each
  if (batch * heads >= kAttnRound) return 0;
  // About one round of equal pieces for the smaller batches, which leaves the
  // least to merge (one request of 32 heads, 32768 tokens: 185 us with 512,
  // 187-191 with 768 to 2048; 256 is 181 there but 197 against 172 for two
  // unequal requests).  From half a round of heads on a request has few
  // pieces, and rounding its share up to whole ones unbalances one round:
  // two (12 requests of 512-2048 tokens: 100 us against 109; unsplit 107).
  // A full round of heads stays unsplit (16 such requests: 118 us, 122 in
  // pieces).  The largest request's pieces bound the room a list of known
  // length uses.
  const long long target = batch * heads <= kAttnRound / 2 ? kAttnRound : 2 * kAttnRound;
  long long room = (target + heads - 1) / heads;
  if (max_slots > 0) room = std::min(room, batch * ((max_slots + shape.align - 1) / shape.align));
  room = std::min<long long>(room, kAttnMaxPieces);
  const long long fit =
      static_cast<long long>(kAttnPieceWords) / (heads * (pool.head_dim + 2)) - batch;
  room = std::min(room, fit);
  return room > 0 ? static_cast<int>(room) : 0;
}

void LaunchAttention(const PoolView& pool, const AttentionArgs& args,
                     hipStream_t stream) {
  if (args.batch <= 0 || pool.num_heads <= 0) return;
  const int D = pool.head_dim;
  if (D <= 0 || D > 256) {
    throw std::invalid_argument("head_dim must be in (0, 256]");
  }
  const long long heads = static_cast<long long>(args.batch) * pool.num_heads;
  const AttnShape shape =
      FastShape(D, args.wide_partition && pool.elements == kFE, heads, args.max_slots);
  if (shape.fn != nullptr) {
    if (args.piece_room < 0 || args.piece_room > kAttnMaxPieces ||
        (args.piece_room > 0 &&
         (shape.split == nullptr || args.piece_words == nullptr ||
          args.piece_arrivals == nullptr || args.piece_tag == 0 ||
          static_cast<long long>(args.batch) * pool.num_heads > kAttnPieceCounters ||
          static_cast<long long>(args.batch + args.piece_room) * pool.num_heads * (D + 2) >
              static_cast<long long>(kAttnPieceWords)))) {
      throw std::invalid_argument("attention pieces do not fit their scratch");
    }
    AttentionArgs a = args;
    a.piece_share = PieceShare(heads) / static_cast<float>(args.batch);
    const dim3 grid(pool.num_heads, args.batch + args.piece_room);
    hipLaunchKernelGGL(a.piece_room > 0 ? shape.split : shape.fn, grid, dim3(shape.waves * kWave),
                       0, stream, pool, a);
    DSD_HIP_CHECK(hipGetLastError());
    return;
  }
  switch (D % 4 == 0 ? D / 4 : 0) {
    case 1: LaunchAttentionT<1>(pool, args, stream); break;
    case 2: LaunchAttentionT<2>(pool, args, stream); break;
    case 4: LaunchAttentionT<4>(pool, args, stream); break;
    case 8: LaunchAttentionT<8>(pool, args, stream); break;
    default: LaunchAttentionT<0>(pool, args, stream); break;
  }
  DSD_HIP_CHECK(hipGetLastError());
}

void PreloadAttentionKernels(const PoolView& pool) {
  for (long long max_slots : {0, 1}) {
    const AttnShape shape = FastShape(pool.head_dim, false, 1, max_slots);
    if (shape.fn == nullptr) continue;
    PreloadKernel(shape.fn);
    if (shape.split != nullptr) PreloadKernel(shape.split);
  }
  if (pool.head_dim == 128 && pool.elements == kFE) PreloadKernel(FastShape(128, true, 1, 0).fn);
}

}  // namespace dsdk
