// attention_head.h -- one head's gather + softmax attention by a workgroup
// (gfx950), shared by the attention kernels (attention.hip) and the wide
// step's attention items (step_kernels.hip).  Reference: GatherPagesCpu +
// SparseAttentionCpu, src/reference_kernels.cpp:109-194.
//
// LPT lanes own one token's D-element head row (D/LPT contiguous dims each,
// float4 loads), a wave covers 64/LPT tokens per chunk and requests UNROLL
// chunks of K and V before it consumes any (bytes in flight per wave =
// UNROLL * 64/LPT * 2 * D * 4); the waves stride over the token slots.  Each
// lane keeps an online softmax (m, l, acc) in the log2 domain (q pre-scaled
// by scale * log2 e, so each exponential is one v_exp_f32); the streams merge
// once at the end, across lanes by xor shuffles and across waves through LDS.
#pragma once

#include "dsd_internal.h"
#include "step_common.h"

namespace dsdk {
namespace {

// The wide step's attention items (D = 128): one head of one request, a whole
// 16-wave workgroup on it, with this lane split; the three-kernel step's
// attention splits the heads of the same batches the same way
// (AttentionArgs::wide_partition), so both step forms give bit-identical
// outputs.  Two heads per item (8 waves each) measured 10 us slower at 32
// requests of 2048 pages: the attention of the requests selected last ends
// later.
constexpr int kWideAttnLpt = 16;
constexpr int kWideAttnWaves = 16;
constexpr int kWideAttnUnroll = 4;

// A stream's maximum before its first token: the lowest float, not -inf, so
// that a logit of -inf weighs exp2(-inf) = 0 also there (-inf - -inf would make
// the stream NaN), with no test in the loop.
constexpr float kNoMax = -0x1.fffffep127f;

template <int WAVES, int D>
struct AttnFastShared {
  float m[WAVES];
  float l[WAVES];
  alignas(16) float acc[WAVES][D];
};

template <int DQ>
struct AttnState {
  float q[DQ];
  float acc[DQ];
  float m, l;
};

// The lane's part of head h's query row, and an empty softmax.
template <int DQ>
__device__ __forceinline__ void AttnBegin(const float* __restrict__ query_row, float scale,
                                          AttnState<DQ>& st) {
  const float qscale = scale * kLog2e;
  LoadDims<DQ>(query_row, st.q);
#pragma unroll
  for (int i = 0; i < DQ; ++i) {
    st.q[i] *= qscale;
    st.acc[i] = 0.0f;
  }
  st.m = kNoMax;
  st.l = 0.0f;
}

// The token slots [f0, f1) of the head's page list (slot f: token f mod
// page_size of list entry f / page_size), wave by wave from f0 in chunks.
// row(s, t, &page): whether token t of list entry s is valid, and its page.
// kPin: keep a row's addresses apart from the registers its loads fill.  Where
// the allocator shares them (it does in the split attention kernel), a chunk's
// loads wait for every load before them.
template <int D, int LPT, int WAVES, int UNROLL, bool kPin = false, class Row>
__device__ __forceinline__ void AttnRange(const PoolView& pool, int head_off, int tid, int f0,
                                          int f1, Row row, AttnState<D / LPT>& st) {
  constexpr int DQ = D / LPT;
  constexpr int TPC = kWave / LPT;
  static_assert(DQ % 4 == 0, "float4 rows");
  const int wave = tid / kWave;
  const int g = (tid & (kWave - 1)) / LPT;
  const int E = pool.elements;
  const int ps = pool.page_size;
  for (int base = f0 + wave * TPC * UNROLL; base < f1; base += WAVES * TPC * UNROLL) {
    float kv[UNROLL][DQ];
    float vv[UNROLL][DQ];
    bool valid[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int f = base + u * TPC + g;
      valid[u] = false;
      if (f < f1) {
        const int slot = f / ps;
        const int t = f - slot * ps;
        int page;
        valid[u] = row(slot, t, &page);
        if (valid[u]) {
          const size_t off = static_cast<size_t>(page) * pool.page_elems +
                             static_cast<size_t>(t) * E + head_off;
          const float* key = pool.keys + off;
          const float* value = pool.values + off;
          LoadDims<DQ>(key, kv[u]);
          LoadDims<DQ>(value, vv[u]);
          if constexpr (kPin) asm volatile("" : : "v"(key), "v"(value));
        }
      }
    }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      float dot = 0.0f;
      if (valid[u]) {
#pragma unroll
        for (int i = 0; i < DQ; ++i) dot = fmaf(st.q[i], kv[u][i], dot);
      }
#pragma unroll
      for (int o = 1; o < LPT; o <<= 1) dot += __shfl_xor(dot, o, kWave);
      if (valid[u]) {
        const float m_new = fmaxf(st.m, dot);
        const float alpha = Exp2(st.m - m_new);
        const float beta = Exp2(dot - m_new);
        st.l = fmaf(st.l, alpha, beta);
#pragma unroll
        for (int i = 0; i < DQ; ++i) st.acc[i] = fmaf(st.acc[i], alpha, beta * vv[u][i]);
        st.m = m_new;
      }
    }
  }
}

// Merges the token streams of each wave and leaves the waves' states in LDS;
// ends with a workgroup barrier.
template <int D, int LPT, int WAVES>
__device__ __forceinline__ void AttnMergeWave(int tid, AttnState<D / LPT>& st,
                                              AttnFastShared<WAVES, D>& sh) {
  constexpr int DQ = D / LPT;
  const int lane = tid & (kWave - 1);
  const int wave = tid / kWave;
  const int g = lane / LPT;
  const int j = lane % LPT;
  float wm = st.m;
#pragma unroll
  for (int o = LPT; o < kWave; o <<= 1) wm = fmaxf(wm, __shfl_xor(wm, o, kWave));
  const float sc = Exp2(st.m - wm);
  float wl = st.l * sc;
#pragma unroll
  for (int i = 0; i < DQ; ++i) st.acc[i] *= sc;
#pragma unroll
  for (int o = LPT; o < kWave; o <<= 1) {
    wl += __shfl_xor(wl, o, kWave);
#pragma unroll
    for (int i = 0; i < DQ; ++i) st.acc[i] += __shfl_xor(st.acc[i], o, kWave);
  }
  if (g == 0) {
    if (j == 0) {
      sh.m[wave] = wm;
      sh.l[wave] = wl;
    }
#pragma unroll
    for (int i = 0; i < DQ; ++i) sh.acc[wave][j * DQ + i] = st.acc[i];
  }
  __syncthreads();
}

// The waves' states in LDS merged: *mx their largest maximum, *lt and *at (dim
// d) their sums relative to it.
template <int D, int WAVES>
__device__ __forceinline__ void AttnCombine(const AttnFastShared<WAVES, D>& sh, int d, float* mx,
                                            float* lt, float* at) {
  float m = kNoMax;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) m = fmaxf(m, sh.m[w]);
  float l = 0.0f, a = 0.0f;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    const float sw = Exp2(sh.m[w] - m);
    l = fmaf(sh.l[w], sw, l);
    a = fmaf(sh.acc[w][d], sw, a);
  }
  *mx = m;
  *lt = l;
  *at = a;
}

// The output of a head's merged sums: zero where no token weighs anything (none
// is valid, or every logit is NaN or -inf).
__device__ __forceinline__ float AttnOutput(float m, float l, float a) {
  return l == 0.0f || (m == kNoMax && !(l > 0.0f)) ? 0.0f : a / l;
}

// Head h of request r over the `count` pages of `list` (global or LDS), by
// WAVES waves whose thread index within the head is tid; holds a workgroup
// barrier (every thread of the workgroup must call it).
template <int D, int LPT, int WAVES, int UNROLL, class List>
__device__ __forceinline__ void AttentionFastHead(const PoolView& pool, const AttentionArgs& args,
                                                  int h, int r, int tid, List list, int count,
                                                  AttnFastShared<WAVES, D>& sh) {
  constexpr int DQ = D / LPT;
  const int head_off = h * D + (tid & (kWave - 1)) % LPT * DQ;
  AttnState<DQ> st;
  AttnBegin<DQ>(args.queries + static_cast<size_t>(r) * pool.elements + head_off, args.scale, st);
  AttnRange<D, LPT, WAVES, UNROLL>(
      pool, head_off, tid, 0, count * pool.page_size,
      [&](int s, int t, int* page) {
        *page = list[s];
        return InPool(*page, pool.capacity) && t < pool.token_counts[*page];
      },
      st);
  AttnMergeWave<D, LPT, WAVES>(tid, st, sh);
  float* out = args.outputs + static_cast<size_t>(r) * pool.elements + static_cast<size_t>(h) * D;
  for (int d = tid; d < D; d += WAVES * kWave) {
    float mx, lt, at;
    AttnCombine<D, WAVES>(sh, d, &mx, &lt, &at);
    out[d] = AttnOutput(mx, lt, at);
  }
}

}  // namespace
}  // namespace dsdk
