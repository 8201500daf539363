#pragma once
// y[M,N] = epilogue(x[M,K] . W[N,K]^T) on fp16 MFMA with fp32 accumulation.
//
// Weights live in HBM in a tile-packed layout (see pack kernels below): the 16 x 32 block of
// W that one v_mfma_f32_16x16x32_f16 consumes as its A operand is one contiguous KB, stored in
// the order the 64 lanes read it, and the blocks of one 16-row tile follow each other along K.
// A wave instruction therefore reads one whole KB and a tile's K sweep is one linear stream.
//
// Six kernels:
//   * stream (M <= 32 packed rows, the decode step; also the fused vocabulary projection +
//     selection of up to 64 rows where the next kernel does not take it): HBM-bound.  A
//     workgroup of 8 waves owns a contiguous range of 16-row tiles (and, with split-K, one K
//     range); it walks the tiles 3 or 4 at a time (1 or 2 where it has no more), the waves taking
//     interleaved K steps.  Activations come in the matching packed fragment layout from L2 and
//     every activation fragment is reused for the tiles of the group.  Fragments are double
//     buffered several steps deep and the prefetch runs across tile-group boundaries, so the
//     memory pipe never drains while a finished group is reduced across the waves through LDS
//     (fixed order: results are run-to-run deterministic).
//   * queues (gemm_queue.h; 33 .. 128 packed rows and 129 .. 256 row-major ones, int8 weights and two row blocks also where
//     a workgroup has five to nine tiles): every wave a K lane with a queue of loads of its own in LDS.
//   * shared-activation stream (vocabularies of 16-bit weights and their selection from one row on; 33 .. 128 packed rows of
//     more tiles than queues take): the same weight streaming, with the activation fragments staged
//     once per workgroup in LDS and shared by its waves.
//   * large tiled, fp16 weights (from 65 row-major rows on): 256 x 256 per workgroup of four waves of
//     128 x 128 with their accumulators in the AGPR bank, both operands global -> LDS directly; tiles of 128 to 256
//     rows and of 64 to 256 columns where the rows are few or leave a round half empty.
//   * large tiled, int8 weights: 256 x 256 x 64 per workgroup of eight waves, weights straight
//     from the packed layout into registers (dequantised there), activations through LDS.
//   * tiled (shapes in between): 128 x 128 x 32 LDS double-buffered tiles, 4 waves of 64 x 64,
//     v_mfma_f32_32x32x16_f16.
// All share one epilogue that reproduces the reference's fp16 rounding points, and a QKV mode
// that scatters K/V into the per-layer cache and scales Q.
#include <math.h>

#include <atomic>
#include <type_traits>
#include <utility>
#include <mutex>

#include "common.h"

enum { MODE_PLAIN = 0, MODE_QKV = 1, MODE_SELECT = 2, MODE_BF = 3, MODE_BF_GLU = 4, MODE_BF_POST = 5 };
// The bf16 modes: operands are bf16 bit patterns (the kernels only move them; what differs is the
// MFMA instruction and the epilogue).  Columns below Epilogue::n32 are stored as bf16, the columns
// from there on as fp32; MODE_BF_GLU stores act(gate, up) of the (gate, up) column pairs below n32;
// MODE_BF_POST is MODE_BF with a bias, an activation and a second output (post4).
template <int MODE>
constexpr bool is_bf = MODE == MODE_BF || MODE == MODE_BF_GLU || MODE == MODE_BF_POST;

struct Epilogue {
  const half_t* bias;
  const half_t* residual;
  half_t* y;
  int N;
  unsigned flags;
  int out_mb;  // > 0: y is written in the packed activation layout with this many 16-row blocks
  // MODE_QKV
  half_t* q_out;
  half_t* Kc;
  half_t* Vc;
  int T, H, hd, S0, S_cap;
  int hd_shift;  // log2(hd) if hd is a power of two, else -1
  const int32_t* len_dev;  // if set (T == 1): per-row append positions on the device (< 0: skip)
  const int32_t* row_dev;  // if set (with len_dev): the row of the cache that each row appends to
  float qscale;
  // MODE_SELECT: greedy selection over the output row instead of (or besides) storing it
  SelectPartial* partials;  // [M][gridDim.x]
  const uint8_t* finished;  // rows that may only emit eos
  const uint8_t* row_mode;  // optional per-row MSA_ROW_* bits
  IdList banned;
  IdList early;  // eos and the stop ids: not eligible for rows with MSA_ROW_BAN_EARLY
  float temperature;  // logits are divided by it when `scale`
  int scale, force_eos_all, eos;
  // bf16 modes
  bf16_t* yb;   // bf16 output, row-major with stride ldy, or packed (out_mb)
  float* y32;   // [M, N - n32] fp32 output of the columns n32 ..
  int n32, ldy;
  int glu;      // MSA_GLU_*
  float limit;  // of MSA_GLU_CLAMPED
  // MODE_BF_POST
  const float* bias32;      // [N] or null
  const float* decay_rate;  // [N - n32] or null: the fp32 columns leave as exp(-rate softplus(z))
  bf16_t* y2;               // bf16 columns from n2 on: row-major with stride ld2, or packed (out2_mb)
  int act, n2, ld2, out2_mb;
};

namespace {

// what MODE_BF_POST does to the sums of columns n .. n + 3, and the vectors it takes for them
struct PostVectors {
  float4_t bias, rate;
};
__device__ __forceinline__ PostVectors post_vectors(const Epilogue& e, int n) {
  PostVectors p{{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  if (e.bias32) p.bias = *reinterpret_cast<const float4_t*>(e.bias32 + n);
  if (n >= e.n32 && e.decay_rate) p.rate = *reinterpret_cast<const float4_t*>(e.decay_rate + n - e.n32);
  return p;
}
__device__ __forceinline__ float4_t post4(const Epilogue& e, int n, float4_t v, const PostVectors& p) {
  v += p.bias;
  if (n < e.n32) {
    if (e.act == MSA_ACT_RELU2) {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = relu2(v[i]);
    }
  } else if (e.decay_rate) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = decay_of(v[i], p.rate[i]);
  }
  return v;
}

// operand fragments of any 16-bit format travel as half8_t
template <int MODE>
__device__ __forceinline__ float4_t mfma_16x16x32(half8_t a, half8_t b, float4_t c) {
  if constexpr (is_bf<MODE>)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
template <int MODE>
__device__ __forceinline__ float16_t mfma_32x32x16(half8_t a, half8_t b, float16_t c) {
  if constexpr (is_bf<MODE>)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// running selection state of one thread for one activation row (see SelectPartial)
struct SelectState {
  float m = -INFINITY, s = 0.f, best = -INFINITY;
  int bidx = 0x7fffffff;
  bool nan = false;
};

// 4 consecutive vocabulary ids n..n+3 of row m: the logit is round(acc), as the stored tensor
// would hold it; log-softmax is monotone, so the arg-max of the masked log-probs is the
// arg-max of the masked logits (lowest id on ties).
__device__ __forceinline__ void select_update4(SelectState& st, const Epilogue& e, int64_t m,
                                               int n, float4_t acc) {
  float z[4], cm = -INFINITY;
  const unsigned rm = e.row_mode ? e.row_mode[m] : 0u;
  const bool only_eos =
      e.force_eos_all || (e.finished && e.finished[m]) || (rm & MSA_ROW_ONLY_EOS);
  const int n_early = (rm & MSA_ROW_BAN_EARLY) ? e.early.n : 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    z[i] = round_h(acc[i]);
    if (e.scale) z[i] = z[i] / e.temperature;
    st.nan |= (z[i] != z[i]);
    cm = fmaxf(cm, z[i]);
    const int id = n + i;
    bool ok = !(only_eos && id != e.eos);
    for (int j = 0; j < e.banned.n; ++j) ok &= (e.banned.id[j] != id);
    for (int j = 0; j < n_early; ++j) ok &= (e.early.id[j] != id);
    const float cand = ok ? z[i] : -INFINITY;
    if (cand > st.best || (cand == st.best && id < st.bidx)) {
      st.best = cand;
      st.bidx = id;
    }
  }
  if (cm > st.m) {
    st.s *= __expf(st.m - cm);
    st.m = cm;
  }
  if (st.m > -INFINITY) {
#pragma unroll
    for (int i = 0; i < 4; ++i) st.s += __expf(z[i] - st.m);
  }
  if (e.y) {
    half4_t o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = (half_t)acc[i];
    *reinterpret_cast<half4_t*>(e.y + m * e.N + n) = o;
  }
}

__device__ __forceinline__ void select_merge(SelectState& a, float om, float os, float ob, int oi,
                                             bool onan) {
  lse_merge(a.m, a.s, om, os);
  if (ob > a.best || (ob == a.best && oi < a.bidx)) {
    a.best = ob;
    a.bidx = oi;
  }
  a.nan |= onan;
}

// What the epilogue of columns n .. n + 3 of row m reads.  A kernel of a few us requests it with its first weights: behind
// its last sum it is a round trip to memory with nothing beside it (qkv and fc1 of a decode step).
template <int MODE>
struct Ahead {
  half4_t bias, res;
  int at, row;  // MODE_QKV: position and row of the cache
  PostVectors post;
};
template <int MODE>
__device__ __forceinline__ Ahead<MODE> epilogue_ahead(const Epilogue& e, int64_t m, int n, bool bias = true) {
  Ahead<MODE> a{};
  if constexpr (MODE == MODE_BF_POST) a.post = post_vectors(e, n);
  if constexpr (is_bf<MODE>) return a;
  if (bias && e.bias) a.bias = *reinterpret_cast<const half4_t*>(e.bias + n);
  if constexpr (MODE == MODE_PLAIN)
    if (e.residual) a.res = *reinterpret_cast<const half4_t*>(e.residual + m * e.N + n);
  if constexpr (MODE == MODE_QKV) {
    const int mi = (int)m;
    a.row = e.T == 1 ? mi : mi / e.T;
    a.at = e.S0;
    if (e.len_dev) {  // per-row lengths: T == 1, row = mi
      a.at = e.len_dev[mi];
      if (e.row_dev) a.row = e.row_dev[mi];
    }
  }
  return a;
}

// 4 consecutive output columns n..n+3 of row m (GIVEN: what it reads is in `a`)
template <int MODE, bool GIVEN = false>
__device__ __forceinline__ void epilogue4(const Epilogue& e, int64_t m, int n, float4_t acc, const Ahead<MODE>& a = {}) {
  if constexpr (is_bf<MODE>) {
    if constexpr (MODE == MODE_BF_POST) acc = post4(e, n, acc, GIVEN ? a.post : post_vectors(e, n));
    if (n >= e.n32) {
      *reinterpret_cast<float4_t*>(e.y32 + m * (e.N - e.n32) + (n - e.n32)) = acc;
    } else if constexpr (MODE != MODE_BF_GLU) {
      const bf16x4_t o = {(bf16_t)acc[0], (bf16_t)acc[1], (bf16_t)acc[2], (bf16_t)acc[3]};
      if (MODE == MODE_BF_POST && n >= e.n2) {
        const int c = n - e.n2;
        *reinterpret_cast<bf16x4_t*>(e.y2 + (e.out2_mb > 0 ? packed_act_offset((int)m, c, e.out2_mb)
                                                           : m * e.ld2 + c)) = o;
        return;
      }
      *reinterpret_cast<bf16x4_t*>(e.yb + (e.out_mb > 0 ? packed_act_offset((int)m, n, e.out_mb)
                                                        : m * e.ldy + n)) = o;
    } else {
      const int c = n >> 1;
      const bf16x2_t o = {(bf16_t)glu_act(e.glu, acc[0], acc[1], e.limit),
                          (bf16_t)glu_act(e.glu, acc[2], acc[3], e.limit)};
      *reinterpret_cast<bf16x2_t*>(e.yb + (e.out_mb > 0 ? packed_act_offset((int)m, c, e.out_mb)
                                                        : m * e.ldy + c)) = o;
    }
    return;
  }
  float t[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) t[i] = round_h(acc[i]);
  if (e.bias) {
    const half4_t b = GIVEN ? a.bias : *reinterpret_cast<const half4_t*>(e.bias + n);
#pragma unroll
    for (int i = 0; i < 4; ++i) t[i] = round_h(t[i] + (float)b[i]);
  }
  if (MODE == MODE_PLAIN) {
    if (e.flags & MSA_EPI_RELU) {
#pragma unroll
      for (int i = 0; i < 4; ++i) t[i] = fmaxf(t[i], 0.f);
    }
    if (e.residual) {
      const half4_t r = GIVEN ? a.res : *reinterpret_cast<const half4_t*>(e.residual + m * e.N + n);
#pragma unroll
      for (int i = 0; i < 4; ++i) t[i] = round_h(t[i] + (float)r[i]);
    }
    half4_t o;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = (half_t)t[i];
    if (e.out_mb > 0)
      *reinterpret_cast<half4_t*>(e.y + packed_act_offset((int)m, n, e.out_mb)) = o;
    else
      *reinterpret_cast<half4_t*>(e.y + m * e.N + n) = o;
  } else {
    // index arithmetic in 32 bits, without 64-bit division: the row count is below 2^31, the
    // thirds are found by comparison, and a power-of-two head size (the usual case) is a shift
    const int D = e.H * e.hd;
    const int part = (n >= D) + (n >= 2 * D), c = n - part * D;  // 0 = K, 1 = V, 2 = Q
    half4_t o;
    if (part == 2) {
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = (half_t)(t[i] * e.qscale);
      *reinterpret_cast<half4_t*>(e.q_out + m * D + c) = o;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = (half_t)t[i];
      const int h = e.hd_shift >= 0 ? c >> e.hd_shift : c / e.hd, d = c - h * e.hd;
      const int mi = (int)m;
      const int b = e.T == 1 ? mi : mi / e.T, tt = mi - b * e.T;
      int s0 = GIVEN ? a.at : e.S0, row = GIVEN ? a.row : b;
      if (!GIVEN && e.len_dev) {  // per-row lengths: T == 1, b = row
        s0 = e.len_dev[b];
        if (e.row_dev) row = e.row_dev[b];
      }
      if (s0 >= 0 && s0 + tt < e.S_cap) {
        half_t* dst = (part == 0 ? e.Kc : e.Vc) +
                      (((int64_t)row * e.H + h) * e.S_cap + s0 + tt) * e.hd + d;
        *reinterpret_cast<half4_t*>(dst) = o;
      }
    }
  }
}

__device__ __forceinline__ half8_t zero8() { return half8_t{0, 0, 0, 0, 0, 0, 0, 0}; }

// 8 packed int8 weights (two dwords) times an fp16 per-row scale -> 8 fp16, each round(q * scale).
// The packed layout stores every byte biased to unsigned (u = q + 128, done once by the pack
// kernel).  u is dropped into the mantissa of fp16 1024.0 (0x6400 | u is exactly 1024 + u) and
// 1152 is subtracted: q exactly, in packed fp16 arithmetic.  The packed multiply then rounds
// the exact product q * scale once, as the fp32 route would.
__device__ __forceinline__ half8_t dequant8(uint32_t lo, uint32_t hi, half_t scale) {
  const half2_t bias = {(half_t)1152.0f, (half_t)1152.0f};
  const half2_t sc = {scale, scale};
  half8_t r;
  const uint32_t w[2] = {lo, hi};
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const uint32_t p0 = __builtin_amdgcn_perm(0x64646464u, w[j], 0x04010400u);  // bytes 0, 1
    const uint32_t p1 = __builtin_amdgcn_perm(0x64646464u, w[j], 0x04030402u);  // bytes 2, 3
    const half2_t h0 = (__builtin_bit_cast(half2_t, p0) - bias) * sc;
    const half2_t h1 = (__builtin_bit_cast(half2_t, p1) - bias) * sc;
    r[4 * j + 0] = h0[0];
    r[4 * j + 1] = h0[1];
    r[4 * j + 2] = h1[0];
    r[4 * j + 3] = h1[1];
  }
  return r;
}

// ---- the tail of a split-K product and the LayerNorm behind it, in front of the next product ----
// Of a few rows every workgroup of the product that follows recomputes x = round(round(round(sum of slices) +
// bias) + x) and LayerNorm(x) for itself, one wave per row, with layernorm_f16_kernel's arithmetic in its
// order (the same bits), while its first weights are on their way.  Bound: a launch of the tail's own costs 3.3 us
// of boundary and a chain of two block-wide sums; here the chain is one wave's, and its operands come out
// of L2.  The first workgroup stores the new residual stream, to another buffer than the one that all read.
constexpr int LN_MAX_ROWS = 8;     // one per wave
constexpr int LN_MAX_K = 2048;     // four 16-byte chunks per lane
template <int S>
struct LnRow {
  static constexpr int C = LN_MAX_K / 512;
  float4_t p[S][C][2];
  half8_t x[C], b[C], g[C], be[C];
  __device__ __forceinline__ void fetch(const LnTail& t, int row, int M, int K, int lane) {
    const int last = (K >> 3) - 1;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if (c > 0 && c * 64 > last) continue;  // uniform
      const int at = min(c * 64 + lane, last) * 8;
#pragma unroll
      for (int i = 0; i < S; ++i) {
        const float* src = t.part + ((int64_t)i * M + row) * K + at;
        p[i][c][0] = *reinterpret_cast<const float4_t*>(src);
        p[i][c][1] = *reinterpret_cast<const float4_t*>(src + 4);
      }
      x[c] = *reinterpret_cast<const half8_t*>(t.x + (int64_t)row * K + at);
      b[c] = *reinterpret_cast<const half8_t*>(t.bias + at);
      g[c] = *reinterpret_cast<const half8_t*>(t.gamma + at);
      be[c] = *reinterpret_cast<const half8_t*>(t.beta + at);
    }
  }
  // (next: what is requested once the slices' registers are free, the second stage of weights: eight rows of 1.3b 1074 ->
  // 1068 us.  In front of the sums it gains nothing more; a wave without a row that skips them costs 90.)
  template <class F>
  __device__ __forceinline__ void finish(const LnTail& t, int row, int M, int K, int lane, bool store,
                                         half_t* rows, F&& next) {
    const int chunks = K >> 3;
    // (the chunks' sums over the wave step by step together: one after the other each waits for itself)
    float sums[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      float s = 0.f;
      sums[c] = 0.f;
      if (c > 0 && c * 64 >= chunks) continue;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float v = p[0][c][i >> 2][i & 3];
#pragma unroll
        for (int k = 1; k < S; ++k) v += p[k][c][i >> 2][i & 3];
        v = round_h(round_h(v) + (float)b[c][i]);
        x[c][i] = (half_t)(v + (float)x[c][i]);
        s += (float)x[c][i];
      }
      sums[c] = c * 64 + lane < chunks ? s : 0.f;
    }
    next();
    wave_sums(sums);
    float total = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c) total += sums[c];
    const float mean = total / (float)K;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      float q = 0.f;
      sums[c] = 0.f;
      if (c > 0 && c * 64 >= chunks) continue;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float d = (float)x[c][i] - mean;
        q += d * d;
      }
      sums[c] = c * 64 + lane < chunks ? q : 0.f;
    }
    wave_sums(sums);
    float var = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c) var += sums[c];
    const float rstd = rsqrtf(var / (float)K + t.eps);
    if (row >= M) return;  // uniform
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int idx = c * 64 + lane;
      if (idx >= chunks) continue;
      if (store) *reinterpret_cast<half8_t*>(t.x_out + (int64_t)row * K + idx * 8) = x[c];
      half8_t o;
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = (half_t)(((float)x[c][i] - mean) * rstd * (float)g[c][i] + (float)be[c][i]);
      *reinterpret_cast<half8_t*>(rows + packed_act_offset(row, idx * 8, 1)) = o;
    }
  }
};

// ---- stream kernel (M <= 64) --------------------------------------------------------------
// MFMA fragments: lane l supplies 8 consecutive K elements (offset 8*(l>>4)) of row (l&15) of
// its operand; A rows are output features n, B rows are activation rows m.  The accumulator
// of lane l holds m = l&15 and n = 4*(l>>4) .. +3.
constexpr int ST_KG = 8;  // waves per workgroup = interleaved K lanes
constexpr int ST_NT = 4;  // weight tiles sharing one activation fragment (<= 32 rows)
constexpr int ST_RN = 4;  // tiles reduced across the waves per pass through LDS

// XR: the activations are row-major ([rows, K], fragments gathered 16 bytes per lane) instead
// of packed; the kernel then handles rows m_off .. m_off + M - 1 of a taller matrix (the ragged
// bottom of a prefill-sized product) and the epilogue sees the global row numbers.
// With more than 32 activation rows the activation fragments (re-read from L2 once per tile
// group) outweigh the weights in cache-fill traffic, so the fp16 kernel lets twice as many
// tiles share each fragment and buffers fewer K steps to stay inside the register file (the
// int8 kernel, whose stage also holds the raw bytes of two K steps, would spill).
template <int MB, bool W8, int MODE, bool XR, int KG, int NT, int U, int LN>
__device__ __forceinline__ void stream_tiles(const half_t* __restrict__ xp, const void* __restrict__ Wp,
                                             const half_t* __restrict__ scales, float* __restrict__ part, int M, int N,
                                             int K, int tiles_per_wg, int ks_per_split, const Epilogue& epi,
                                             int64_t m_off, const LnTail& ln) {
  static_assert(LN == 0 || (MB == 1 && !XR && KG == LN_MAX_ROWS), "one wave per row");
  // U = K steps (32 wide) buffered per stage; an int8 block covers two steps
  constexpr int UA = W8 ? U / 2 : U;  // weight loads per stage and tile
  constexpr int RN = NT < ST_RN ? NT : ST_RN;  // NT is a multiple of RN
  __shared__ float4_t red[KG][RN * MB][64];
  extern __shared__ __attribute__((aligned(16))) half_t ln_rows[];  // LN: the normed rows, packed (one row block)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ntiles = N >> 4;
  const int nks = K >> 5;  // 32-wide steps in a row
  const int tile_begin = blockIdx.x * tiles_per_wg;
  const int tile_end = min(ntiles, tile_begin + tiles_per_wg);
  const int ks_begin = blockIdx.y * ks_per_split;
  const int ks_end = min(nks, ks_begin + ks_per_split);
  if (tile_begin >= tile_end || ks_begin >= ks_end) return;
  const int ngroups = (tile_end - tile_begin + NT - 1) / NT;
  const int nstages = (ks_end - ks_begin + KG * U - 1) / (KG * U);
  const int total = ngroups * nstages;
  // A stage is followed, not found by division: 30 scalar instructions each time, in kernels of a few us (int8, one row, 6144
  // x 2048 5.0 and 4.8 us).  Of three or four int8 tiles to a group the division is ahead, whose operands take fewer
  // registers through the loop: 36864 x 9216 59.2 and 57.5, 28672 x 7168 38.2 and 37.2, 15360 x 5120 15.7 and 15.0.
  constexpr bool BY_INDEX = W8 && NT > 2;
  struct At {
    int n, st, nstages;  // n: the group, or (BY_INDEX) the stage counted over all groups
    __device__ void next() {
      if (BY_INDEX)
        ++n;
      else if (++st == nstages)
        st = 0, ++n;
    }
    __device__ bool last() const { return BY_INDEX ? (n + 1) % nstages == 0 : st + 1 == nstages; }
  };

  // In the last row block the lanes of rows past M read row M - 1 (what they add is not stored): half as many lines to fetch
  // for eight rows, a quarter and less for fewer.  4 rows, us: 2048 x 8192 11.5 -> 9.9, 4096 x 4096 7.5 -> 7.0; with three or
  // four tiles to an activation fragment the weights' lines are what counts, and it costs 1 to 2 % (12288 x 4096 16.2, 16.5).
  const int last_lane = NT > 2 ? lane : (lane & 48) + min(lane & 15, M - 1 - (MB - 1) * 16);

  struct Stage {
    half8_t a[UA][NT];  // fp16: one A fragment; int8: 16 raw bytes = two A fragments
    half8_t b[U][MB];
  };
  Stage s0, s1;
  // Loads are unconditional so that the hardware counters can keep two stages in flight (a
  // load inside a branch makes the compiler wait for every outstanding load before the MFMAs).
  // Steps and tiles past the end read a clamped, valid address: a surplus tile is dropped in
  // finish(), a surplus step gets its activation fragment zeroed in mma().
  auto load = [&](Stage& s, const At& at) {
    const int grp = BY_INDEX ? at.n / nstages : at.n, st = BY_INDEX ? at.n - grp * nstages : at.st;
    const int t0 = tile_begin + grp * NT;
#pragma unroll
    for (int u = 0; u < UA; ++u) {
      // first 32-wide step covered by this load (wave-uniform)
      const int ks = W8 ? ks_begin + 2 * (wave + KG * (st * UA + u))
                        : ks_begin + wave + KG * (st * U + u);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int t = min(t0 + j, tile_end - 1);
        const int ksc = min(ks, ks_end - (W8 ? 2 : 1));
        const int64_t blk = W8 ? (int64_t)t * (nks >> 1) + (ksc >> 1) : (int64_t)t * nks + ksc;
        s.a[u][j] = __builtin_nontemporal_load(
            reinterpret_cast<const half8_t*>((const half_t*)Wp + blk * 512 + lane * 8));
      }
      if constexpr (LN > 0) continue;  // the activations are in LDS
#pragma unroll
      for (int h = 0; h < (W8 ? 2 : 1); ++h) {
        const int kk = min(ks + h, ks_end - 1);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
          if (XR) {
            const int64_t m = m_off + min(mb * 16 + (lane & 15), M - 1);
            s.b[W8 ? 2 * u + h : u][mb] = *reinterpret_cast<const half8_t*>(
                xp + m * K + kk * 32 + (lane >> 4) * 8);
          } else {
            s.b[W8 ? 2 * u + h : u][mb] = *reinterpret_cast<const half8_t*>(
                xp + (((int64_t)kk * MB + mb) * 64 + (mb + 1 < MB ? lane : last_lane)) * 8);
          }
        }
      }
    }
  };
  // slot e = threadIdx.x + it * KG * 64 of a reduction pass of finish(); it always maps to the
  // same activation row, whatever the pass (MODE_SELECT keeps one running state per slot)
  constexpr int SEL_IT = (RN * MB * 64 + KG * 64 - 1) / (KG * 64);
  SelectState sel[MODE == MODE_SELECT ? SEL_IT : 1];
  float4_t acc[NT][MB];
  auto clear = [&]() {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) acc[j][mb] = float4_t{0.f, 0.f, 0.f, 0.f};
  };
  auto mma = [&](Stage& s, const At& at) {
    const int grp = BY_INDEX ? at.n / nstages : at.n, st = BY_INDEX ? at.n - grp * nstages : at.st;
    half_t sc[NT];
    if (W8) {
      const int t0 = tile_begin + grp * NT;
#pragma unroll
      for (int j = 0; j < NT; ++j)
        sc[j] = scales[min(t0 + j, tile_end - 1) * 16 + (lane & 15)];
    }
    // zero the activation fragments of steps past the end of this K range
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int ks = W8 ? ks_begin + 2 * (wave + KG * (st * UA + u / 2)) + (u & 1)
                        : ks_begin + wave + KG * (st * U + u);
      if constexpr (LN > 0)
        s.b[u][0] = *reinterpret_cast<const half8_t*>(ln_rows + (min(ks, ks_end - 1) * 64 + lane) * 8);
      if (ks >= ks_end) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) s.b[u][mb] = zero8();
      }
    }
    const int tiles_left = tile_end - (tile_begin + grp * NT);  // real tiles in this group
#pragma unroll
    for (int u = 0; u < UA; ++u)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        if (NT > ST_NT && j >= tiles_left) continue;  // wave-uniform: no MFMAs for surplus tiles
        if (!W8) {
#pragma unroll
          for (int mb = 0; mb < MB; ++mb)
            acc[j][mb] = mfma_16x16x32<MODE>(s.a[u][j], s.b[u][mb], acc[j][mb]);
        } else {
          typedef uint32_t u4 __attribute__((ext_vector_type(4)));
          const u4 raw = __builtin_bit_cast(u4, s.a[u][j]);
          const half8_t f0 = dequant8(raw[0], raw[1], sc[j]);
          const half8_t f1 = dequant8(raw[2], raw[3], sc[j]);
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) {
            acc[j][mb] =
                __builtin_amdgcn_mfma_f32_16x16x32_f16(f0, s.b[2 * u][mb], acc[j][mb], 0, 0, 0);
            acc[j][mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f1, s.b[2 * u + 1][mb],
                                                                acc[j][mb], 0, 0, 0);
          }
        }
      }
  };
  // the epilogue's operands of the group that comes next, where a thread has one slot of it (not of int8 weights, whose
  // expansion fills the registers: one row, 12288 x 4096 11.3 and 10.8 us, 5120 x 20480 29.7 and 28.4)
  constexpr bool AHEAD = MB <= 2 && !XR && MODE != MODE_SELECT && (!W8 || LN > 0);
  static_assert(!AHEAD || (SEL_IT == 1 && NT == RN), "one slot");
  constexpr int EMODE = MODE == MODE_SELECT ? MODE_PLAIN : MODE;
  Ahead<EMODE> ahead{};
  auto look_ahead = [&](int grp) {
    if (!AHEAD || part) return;
    const int jm = min((int)threadIdx.x >> 6, RN * MB - 1), jj = jm / MB, mb = jm - jj * MB;
    ahead = epilogue_ahead<EMODE>(epi, min(mb * 16 + (lane & 15), M - 1),
                                  min(tile_begin + grp * NT + jj, tile_end - 1) * 16 + ((lane >> 4) << 2));
  };
  auto finish = [&](int grp) {  // after the last stage of a tile group
    const int t0 = tile_begin + grp * NT;
#pragma unroll
    for (int p = 0; p < NT / RN; ++p) {  // RN tiles per pass through the LDS buffer
#pragma unroll
      for (int jj = 0; jj < RN; ++jj)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) red[wave][jj * MB + mb][lane] = acc[p * RN + jj][mb];
      __syncthreads();
#pragma unroll
      for (int it = 0; it < SEL_IT; ++it) {
        const int e = threadIdx.x + it * KG * 64;
        if (e >= RN * MB * 64) break;
        const int jm = e >> 6, l = e & 63;
        const int jj = jm / MB, mb = jm - jj * MB;
        const int j = p * RN + jj;
        float4_t sum = red[0][jm][l];
#pragma unroll
        for (int w = 1; w < KG; ++w) sum += red[w][jm][l];
        const int m = mb * 16 + (l & 15);
        const int n = (t0 + j) * 16 + ((l >> 4) << 2);
        if (m < M && t0 + j < tile_end) {
          if (part)
            *reinterpret_cast<float4_t*>(part + ((int64_t)blockIdx.y * M + m) * N + n) = sum;
          else if (MODE == MODE_SELECT)
            select_update4(sel[it], epi, m, n, sum);
          else if constexpr (AHEAD)
            epilogue4<EMODE, true>(epi, m_off + m, n, sum, ahead);
          else
            epilogue4<EMODE>(epi, m_off + m, n, sum);
        }
      }
      __syncthreads();
    }
    clear();
    if (grp + 1 < ngroups) look_ahead(grp + 1);
  };
  clear();
  At la{0, 0, nstages}, ma{0, 0, nstages};  // the stages loaded and multiplied next
  if constexpr (LN > 0) {
    // Requested in this order, the tail's operands arrive while the first weights are on their way.
    LnRow<LN> row;
    row.fetch(ln, min(wave, M - 1), M, K, lane);
    load(s0, la);
    look_ahead(0);
    row.finish(ln, wave, M, K, lane, blockIdx.x == 0, ln_rows, [&] {
      if (total > 1) {
        la.next();
        load(s1, la);
      }
    });
    __syncthreads();
  } else {
    load(s0, la);
    look_ahead(0);
  }
  auto take = [&](Stage& s) {
    mma(s, ma);
    if (ma.last()) finish(BY_INDEX ? ma.n / nstages : ma.n);
    ma.next();
  };
  // stage idx is in `a`; steady state: every load is of a real stage
  auto rest = [&](int idx, Stage& a, Stage& b) {
    for (; idx + 2 < total; idx += 2) {
      la.next();
      load(b, la);
      take(a);
      la.next();
      load(a, la);
      take(b);
    }
    if (idx + 1 < total) {  // two stages left
      la.next();
      load(b, la);
      take(a);
      take(b);
    } else {  // one stage left
      take(a);
    }
  };
  if constexpr (LN > 0) {
    take(s0);
    if (total > 1) rest(1, s1, s0);
  } else {
    rest(0, s0, s1);
  }
  if (MODE == MODE_SELECT) {
    // The 16 threads that hold one row (4 lane groups x RN tile slots of one row block) merge
    // their states: lanes through shuffles, tile slots through LDS; one partial per row and
    // workgroup goes to memory for the combine kernel.
    SelectPartial* sp = reinterpret_cast<SelectPartial*>(&red[0][0][0]);  // [RN * MB * 16]
#pragma unroll
    for (int it = 0; it < SEL_IT; ++it) {
      const int e = threadIdx.x + it * KG * 64;
      SelectState st = sel[it];
#pragma unroll
      for (int o = 16; o <= 32; o <<= 1)
        select_merge(st, __shfl_xor(st.m, o, MSA_WAVE), __shfl_xor(st.s, o, MSA_WAVE),
                     __shfl_xor(st.best, o, MSA_WAVE), __shfl_xor(st.bidx, o, MSA_WAVE),
                     (bool)__shfl_xor((int)st.nan, o, MSA_WAVE));
      if (e < RN * MB * 64 && (e & 63) < 16) {
        SelectPartial p;
        p.m = st.m, p.s = st.s, p.best = st.best, p.bidx = st.bidx, p.nan = st.nan ? 1.f : 0.f;
        sp[(e >> 6) * 16 + (e & 15)] = p;  // [jm][row in block]
      }
    }
    __syncthreads();
    if (threadIdx.x < MB * 16) {
      const int mb = threadIdx.x >> 4, r = threadIdx.x & 15;
      SelectState st;
      for (int j = 0; j < RN; ++j) {  // jm = j * MB + mb
        const SelectPartial p = sp[(j * MB + mb) * 16 + r];
        select_merge(st, p.m, p.s, p.best, p.bidx, p.nan > 0.f);
      }
      const int m = mb * 16 + r;
      if (m < M) {
        SelectPartial p;
        p.m = st.m, p.s = st.s, p.best = st.best, p.bidx = st.bidx, p.nan = st.nan ? 1.f : 0.f;
        p.pad[0] = p.pad[1] = p.pad[2] = 0.f;
        epi.partials[(int64_t)m * gridDim.x + blockIdx.x] = p;
      }
    }
  }
}

template <int MB, bool W8, int MODE, bool XR = false, int KG = ST_KG,
          int NT = (MB <= 2 || W8 ? ST_NT : 2 * ST_NT), int U = (MB <= 2 ? 4 : (NT > ST_NT ? 1 : 2))>
__global__ __launch_bounds__(KG * 64) void linear_stream_kernel(
    const half_t* __restrict__ xp, const void* __restrict__ Wp, const half_t* __restrict__ scales,
    float* __restrict__ part, int M, int N, int K, int tiles_per_wg, int ks_per_split, Epilogue epi, int64_t m_off) {
  stream_tiles<MB, W8, MODE, XR, KG, NT, U, 0>(xp, Wp, scales, part, M, N, K, tiles_per_wg, ks_per_split, epi, m_off,
                                               LnTail{});
}

// LN slices' tail and the LayerNorm in front.  What the first loads need is in the first 14 words of the arguments, which
// a wave finds in its registers (nk: N / 16 above 8 bits of K / 32; mt: tiles per workgroup above 8 bits of M).
template <bool W8, int MODE, int NT, int LN>
__global__ __launch_bounds__(ST_KG * 64) void linear_stream_ln_kernel(
    const float* __restrict__ ln_part, const half_t* __restrict__ ln_x, const void* __restrict__ Wp,
    const half_t* __restrict__ ln_bias, const half_t* __restrict__ gamma, const half_t* __restrict__ beta, uint32_t nk,
    uint32_t mt, half_t* __restrict__ x_out, const half_t* __restrict__ scales, float eps, Epilogue epi) {
  const int nks = nk & 255;
  stream_tiles<1, W8, MODE, false, ST_KG, NT, 4, LN>(nullptr, Wp, scales, nullptr, mt & 255, (int)(nk >> 8) * 16, nks * 32,
                                                     mt >> 8, W8 ? (nks + 1) & ~1 : nks, epi, 0,
                                                     LnTail{ln_part, ln_bias, ln_x, x_out, gamma, beta, eps});
}

// ---- shared-activation stream kernel (vocabularies from one row on; more tiles than queues take) ----
// With more than 32 activation rows a wave that loads its own activation fragments moves more
// bytes of activations (from L2) than of weights (from HBM) through the L1, and the L1 fill rate
// becomes the limit.  Here the waves form KL K lanes x NG tile lanes: the NG waves of a K lane
// work on different weight tiles over the same K steps and read their activation fragments from
// LDS, which the whole workgroup fills once per stage (SK = KL * U consecutive K steps, one
// contiguous piece of the packed activations).  Weights still go from HBM straight to registers.
// A tile group is NG * NT tiles, dealt round robin to the tile lanes; one barrier per stage;
// activations are fetched two stages ahead and parked in LDS one stage ahead, weights (and int8
// scales) PF - 1 stages ahead.  The K lanes are summed through LDS in fixed order.
template <int MB, bool W8, int KL, int NG, int NT, int U>
struct ShareCfg {
  static constexpr int THREADS = KL * NG * 64;
  static constexpr int SK = KL * U, UA = W8 ? U / 2 : U;
  static constexpr int XH = SK * MB * 512;  // halves of activations per stage
  static constexpr int PIECES = XH / 8;     // 16-byte pieces per stage
  static constexpr int XP = (PIECES + THREADS - 1) / THREADS;  // pieces per thread and stage
  // activations double buffered, then one tile slot's partial sums of the other K lanes
  static constexpr int RED_BYTES = (KL - 1) * NG * MB * 1024;
  static constexpr int LDS_BYTES = 2 * XH * 2 + RED_BYTES;
  static_assert(LDS_BYTES <= 160 * 1024, "a CU has 160 KB of LDS");
  static_assert(U % 2 == 0, "a stage holds whole int8 blocks");
};

template <int MB, bool W8, int MODE, int KL, int NG, int NT, int U, int PF>
__global__ __launch_bounds__(KL * NG * 64) void linear_share_kernel(
    const half_t* __restrict__ xp, const void* __restrict__ Wp, const half_t* __restrict__ scales,
    float* __restrict__ part, int M, int N, int K, int tiles_per_wg, int ks_per_split,
    Epilogue epi) {
  static_assert(MODE != MODE_SELECT || (KL == 1 && NT == 1), "a wave that selects owns its tiles' sums");
  using C = ShareCfg<MB, W8, KL, NG, NT, U>;
  constexpr int SK = C::SK, UA = C::UA, XH = C::XH, XP = C::XP, THREADS = C::THREADS;
  constexpr int PIECES = C::PIECES;
  extern __shared__ __attribute__((aligned(16))) half_t lx_share[];  // [2][XH], then red
  float4_t* red = reinterpret_cast<float4_t*>(lx_share + 2 * XH);  // [KL-1][NG][MB][64]
  const int lane = threadIdx.x & 63;
  // the wave number as a scalar: everything derived from it stays out of the vector registers
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kl = wave / NG, ng = wave - kl * NG;
  const uint32_t lane_off = (uint32_t)lane * 16u;  // the lane's 16 bytes of a 1 KB fragment
  const int ntiles = N >> 4, nks = K >> 5;
  const int tile_begin = blockIdx.x * tiles_per_wg;
  const int tile_end = min(ntiles, tile_begin + tiles_per_wg);
  const int ks_begin = blockIdx.y * ks_per_split;
  const int ks_end = min(nks, ks_begin + ks_per_split);
  if (tile_begin >= tile_end || ks_begin >= ks_end) return;
  const int ngroups = (tile_end - tile_begin + NG * NT - 1) / (NG * NT);
  const int nstages = (ks_end - ks_begin + SK - 1) / SK;
  const int total = ngroups * nstages;

  // Every load is unconditional (clamped address): K steps past the end are zeroed on their way
  // into LDS, tiles past the end are dropped in finish().
  half8_t xr[XP];
  auto gload_x = [&](int idx) {
    const int kb = ks_begin + (idx % nstages) * SK;
#pragma unroll
    for (int i = 0; i < XP; ++i) {
      // Piece p = 64 * f + lane: fragment f is the same for the whole wave, so the address is a
      // scalar base plus the lane's 16 bytes.  A stage need not split evenly over the waves:
      // surplus slots re-read the last fragment.
      const int f = min(wave + (THREADS / 64) * i, PIECES / 64 - 1);
      const int kk = min(kb + f / MB, ks_end - 1);
      const half_t* frag = xp + ((int64_t)kk * MB + f % MB) * 512;
      xr[i] = *reinterpret_cast<const half8_t*>(reinterpret_cast<const char*>(frag) + lane_off);
    }
  };
  auto lstore = [&](int idx) {
    const int kb = ks_begin + (idx % nstages) * SK;
    half_t* l = lx_share + (idx & 1) * XH;
#pragma unroll
    for (int i = 0; i < XP; ++i) {
      const int f = wave + (THREADS / 64) * i;  // wave-uniform, as are the two conditions
      const bool live = kb + f / MB < ks_end;
      if (PIECES % THREADS == 0 || f < PIECES / 64)
        *reinterpret_cast<half8_t*>(l + f * 512 + lane * 8) = live ? xr[i] : zero8();
    }
  };
  struct Wst {
    half8_t a[UA][NT];  // fp16: one A fragment; int8: 16 raw bytes = two A fragments
  };
  uint32_t sc[NT];  // int8: the row's fp16 scale in the low half, one per tile of the group
  auto gload_sc = [&](int grp) {
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int t = min(tile_begin + (grp * NT + j) * NG + ng, tile_end - 1);
      sc[j] = W8 ? reinterpret_cast<const uint16_t*>(scales)[t * 16 + (lane & 15)] : 0u;
    }
  };
  auto gload_w = [&](Wst& w, int idx) {
    const int grp = idx / nstages, st = idx - grp * nstages;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int t = min(tile_begin + (grp * NT + j) * NG + ng, tile_end - 1);
#pragma unroll
      for (int u = 0; u < UA; ++u) {
        const int ks = ks_begin + st * SK + kl * U + (W8 ? 2 * u : u);
        const int ksc = min(ks, ks_end - (W8 ? 2 : 1));
        const int64_t blk = W8 ? (int64_t)t * (nks >> 1) + (ksc >> 1) : (int64_t)t * nks + ksc;
        const half_t* block = (const half_t*)Wp + blk * 512;  // wave-uniform
        w.a[u][j] = __builtin_nontemporal_load(
            reinterpret_cast<const half8_t*>(reinterpret_cast<const char*>(block) + lane_off));
      }
    }
  };

  // A wave that owns all of its tiles' K sums every stage by itself and then the stages, where the sums leave in 32 bits:
  // one chain over all of K had two to three times the error of sums over eight waves (bf16 of K = 768 / 2048 / 4096 /
  // 9216: 1.6 / 2.7 / 3.9 / 6.1e-7, eight waves 0.8 / 1.0 / 1.4 / 2.0e-7, so 0.8 / 1.0 / 1.2 / 1.7e-7, at no cost in time).
  // Results of 16 bits are the same to five digits either way.  More row blocks leave no registers for it (launch_wide).
  constexpr bool LEVELS = KL == 1 && MB <= 4 && MODE != MODE_SELECT;
  float4_t acc[NT][MB], done[LEVELS ? NT : 1][LEVELS ? MB : 1];
  auto clear = [&]() {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        acc[j][mb] = float4_t{0.f, 0.f, 0.f, 0.f};
        if (LEVELS) done[LEVELS ? j : 0][LEVELS ? mb : 0] = acc[j][mb];
      }
  };
  auto settle = [&]() {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        done[LEVELS ? j : 0][LEVELS ? mb : 0] += acc[j][mb];
        acc[j][mb] = float4_t{0.f, 0.f, 0.f, 0.f};
      }
  };
  auto sum_of = [&](int j, int mb) {
    return LEVELS ? done[LEVELS ? j : 0][LEVELS ? mb : 0] + acc[j][mb] : acc[j][mb];
  };
  auto compute = [&](const Wst& w, int idx) {
    const half_t* l = lx_share + (idx & 1) * XH + kl * U * MB * 512 + lane * 8;
    constexpr int F = U * MB;  // fragment f = K step f / MB, row block f % MB
    constexpr int PD = KL * NG > 8 ? 2 : 4;  // LDS fragment reads in flight (registers are
                                             // scarcer at three waves per SIMD)
    half8_t bx[PD];
#pragma unroll
    for (int p = 0; p < PD; ++p) bx[p] = *reinterpret_cast<const half8_t*>(l + p * 512);
    // the A fragments of K step u (one set only where registers are scarce: the other waves of
    // the SIMD then cover the expansion)
    constexpr int AB = PF > 2 ? 1 : 2;
    half8_t a[AB][NT];
    auto expand = [&](int u) {
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        if (W8) {
          typedef uint32_t u4 __attribute__((ext_vector_type(4)));
          const u4 raw = __builtin_bit_cast(u4, w.a[u / 2][j]);
          const half_t scj = __builtin_bit_cast(half2_t, sc[j])[0];
          a[u % AB][j] = (u & 1) ? dequant8(raw[2], raw[3], scj) : dequant8(raw[0], raw[1], scj);
        } else {
          a[u % AB][j] = w.a[W8 ? 0 : u][j];
        }
      }
    };
    // the stage's LDS stores and global loads go out first, then LDS reads and MFMAs alternate
    __builtin_amdgcn_sched_group_barrier(0x200, XP, 0);
    __builtin_amdgcn_sched_group_barrier(0x020, XP, 0);  // activations first: needed first
    __builtin_amdgcn_sched_group_barrier(0x020, UA * NT, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, PD, 0);
#pragma unroll
    for (int f = 0; f < F; ++f) {
      const int u = f / MB, mb = f % MB;
      if (mb == 0) expand(u);
      const half8_t cur = bx[f % PD];
#pragma unroll
      for (int j = 0; j < NT; ++j)
        acc[j][mb] = mfma_16x16x32<MODE>(a[u % AB][j], cur, acc[j][mb]);
      __builtin_amdgcn_sched_group_barrier(0x008, NT, 0);
      if (f + PD < F) {
        bx[f % PD] = *reinterpret_cast<const half8_t*>(l + (f + PD) * 512);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
    }
  };
  SelectState sel[MODE == MODE_SELECT ? MB : 1];  // of row lane % 16 of each block
  auto finish = [&](int idx) {  // after the last stage of a tile group
    const int grp = idx / nstages;
    if constexpr (MODE == MODE_SELECT) {
      const int t = tile_begin + grp * NG + ng;
      if (t < tile_end) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          if (mb * 16 + (lane & 15) < M)
            select_update4(sel[mb], epi, mb * 16 + (lane & 15), t * 16 + ((lane >> 4) << 2), sum_of(0, mb));
      }
      clear();
      return;
    }
    constexpr int EMODE = MODE == MODE_SELECT ? MODE_PLAIN : MODE;
    // What the epilogue reads is requested for all row blocks at once, in front of the reduction (row by row behind it, each
    // block is a round trip), where there are registers for it: of eight row blocks they spill; int8 weights and a cache to
    // write to lose the loads in flight by it (int8, 40 rows in slices, 7168 x 28672 52.7 without and 56.8 us with it).
    constexpr bool AHEAD = MB <= 4 && EMODE == MODE_PLAIN && !W8;
    Ahead<EMODE> ahead[AHEAD ? MB : 1];
    auto look_ahead = [&](int t) {
      if (!AHEAD || part || kl > 0) return;
      const int n = min(t, tile_end - 1) * 16 + ((lane >> 4) << 2);
#pragma unroll
      for (int mb = 0; mb < (AHEAD ? MB : 0); ++mb) {
        ahead[mb] = epilogue_ahead<EMODE>(epi, min(mb * 16 + (lane & 15), M - 1), n, mb == 0);
        ahead[mb].bias = ahead[0].bias;
      }
    };
#pragma unroll
    for (int j = 0; j < NT; ++j) {  // one tile slot per round through the reduction buffer
      look_ahead(tile_begin + (grp * NT + j) * NG + ng);
      if (kl > 0) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          red[(((kl - 1) * NG + ng) * MB + mb) * 64 + lane] = acc[j][mb];
      }
      __syncthreads();
      const int t = tile_begin + (grp * NT + j) * NG + ng;
      if (kl == 0 && t < tile_end) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
          float4_t sum = sum_of(j, mb);
#pragma unroll
          for (int k = 1; k < KL; ++k) sum += red[(((k - 1) * NG + ng) * MB + mb) * 64 + lane];
          const int m = mb * 16 + (lane & 15);
          const int n = t * 16 + ((lane >> 4) << 2);
          if (m >= M) continue;
          if (part)
            *reinterpret_cast<float4_t*>(part + ((int64_t)blockIdx.y * M + m) * N + n) = sum;
          else
            epilogue4<EMODE, AHEAD>(epi, m, n, sum, ahead[AHEAD ? mb : 0]);
        }
      }
      if (j + 1 < NT) __syncthreads();  // the buffer is rewritten by the next slot
    }
    clear();
    if (W8 && grp + 1 < ngroups) gload_sc(grp + 1);
  };

  // PF - 1 weight stages in flight beyond the one being consumed
  Wst w[PF];
  clear();
  if (W8) gload_sc(0);
  // same issue order as in the loop (activations of the next stage, then weights), so that the
  // wait before the loop's first LDS store does not cover the weight loads
  gload_x(0);
  lstore(0);
  gload_x(1);
#pragma unroll
  for (int st = 0; st < PF - 1; ++st) gload_w(w[st], st);
  __syncthreads();
  // Stages are taken PF at a time; surplus stages at the end work on clamped addresses into
  // accumulators that are never stored.
  for (int idx = 0; idx < total; idx += PF) {
#pragma unroll
    for (int st = 0; st < PF; ++st) {
      const int i = idx + st;
      lstore(i + 1);  // fetched during stage i - 1
      gload_x(i + 2);
      gload_w(w[(st + PF - 1) % PF], i + PF - 1);
      compute(w[st], i);
      if (LEVELS && (is_bf<MODE> || part)) settle();
      if (i < total && (i + 1) % nstages == 0) finish(i);
      __syncthreads();
    }
  }
  if constexpr (MODE == MODE_SELECT) {  // the row's lanes through shuffles, the waves through LDS, as in the stream kernel
    static_assert(NG * MB * 16 * sizeof(SelectPartial) <= C::LDS_BYTES, "the states take the stages' place");
    SelectPartial* sp = reinterpret_cast<SelectPartial*>(lx_share);  // [NG][MB * 16]
    auto partial_of = [](const SelectState& st) {
      SelectPartial p;
      p.m = st.m, p.s = st.s, p.best = st.best, p.bidx = st.bidx, p.nan = st.nan ? 1.f : 0.f;
      p.pad[0] = p.pad[1] = p.pad[2] = 0.f;
      return p;
    };
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      SelectState st = sel[mb];
#pragma unroll
      for (int o = 16; o <= 32; o <<= 1)
        select_merge(st, __shfl_xor(st.m, o, MSA_WAVE), __shfl_xor(st.s, o, MSA_WAVE),
                     __shfl_xor(st.best, o, MSA_WAVE), __shfl_xor(st.bidx, o, MSA_WAVE),
                     (bool)__shfl_xor((int)st.nan, o, MSA_WAVE));
      if (lane < 16) sp[ng * (MB * 16) + mb * 16 + lane] = partial_of(st);
    }
    __syncthreads();
    const int m = threadIdx.x;
    if (m < MB * 16 && m < M) {
      SelectState st;
      for (int w = 0; w < NG; ++w) {
        const SelectPartial p = sp[w * (MB * 16) + m];
        select_merge(st, p.m, p.s, p.best, p.bidx, p.nan > 0.f);
      }
      epi.partials[(int64_t)m * gridDim.x + blockIdx.x] = partial_of(st);
    }
  }
}

// sums split-K partials part[s][m][n] in slice order and applies the epilogue
template <int MODE>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ part, int S,
                                                            int M, int N, Epilogue epi) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;  // one float4 of one row
  const int nq = N >> 2;
  if (idx >= (int64_t)M * nq) return;
  const int m = (int)(idx / nq), n = (int)(idx % nq) << 2;
  float4_t s = *reinterpret_cast<const float4_t*>(part + (int64_t)m * N + n);
  for (int i = 1; i < S; ++i)
    s += *reinterpret_cast<const float4_t*>(part + ((int64_t)i * M + m) * N + n);
  epilogue4<MODE>(epi, m, n, s);
}

// ---- tiled kernel ---------------------------------------------------------------------
constexpr int TL_BM = 128, TL_BN = 128, TL_BK = 32, TL_LD = TL_BK + 8, TL_THREADS = 256;

template <bool W8, int MODE>
__global__ __launch_bounds__(TL_THREADS) void linear_tiled_kernel(
    const half_t* __restrict__ x, const void* __restrict__ Wp, const half_t* __restrict__ scales,
    int64_t M, int N, int K, Epilogue epi) {
  __shared__ __attribute__((aligned(16))) half_t lx[2][TL_BM * TL_LD];
  __shared__ __attribute__((aligned(16))) half_t lw[2][TL_BN * TL_LD];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  const int li = lane & 31, lg = lane >> 5;
  const int64_t m0 = (int64_t)blockIdx.y * TL_BM;
  const int n0 = blockIdx.x * TL_BN;
  const int nkt = K / TL_BK;
  const int nks = K >> 5;

  // staging: each thread moves two 16-byte pieces of each operand tile.  x: piece c covers row
  // c/4, columns 8*(c%4); W: piece c is lane c%64 of the packed block of row tile c/64.
  int xrow[2], xcol[2], wrow[2], wcol[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int c = tid + TL_THREADS * i;
    xrow[i] = c >> 2;
    xcol[i] = (c & 3) << 3;
    wrow[i] = (c >> 6) * 16 + (c & 15);
    wcol[i] = ((c >> 4) & 3) << 3;
  }
  half8_t rx[2], rw[2];

  auto load_tile = [&](int kt) {
    const int k0 = kt * TL_BK;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int64_t m = m0 + xrow[i];
      if (m < M)
        rx[i] = *reinterpret_cast<const half8_t*>(x + m * K + k0 + xcol[i]);
      else
        rx[i] = zero8();
      const int n = n0 + wrow[i];
      if (n < N) {
        const int c = tid + TL_THREADS * i;
        if (!W8) {
          rw[i] = *reinterpret_cast<const half8_t*>((const half_t*)Wp +
                                                    ((int64_t)(n >> 4) * nks + kt) * 512 +
                                                    (c & 63) * 8);
        } else {
          const uint2 w = *reinterpret_cast<const uint2*>(
              (const int8_t*)Wp + ((int64_t)(n >> 4) * (nks >> 1) + (kt >> 1)) * 1024 +
              (c & 63) * 16 + (kt & 1) * 8);
          rw[i] = dequant8(w.x, w.y, scales[n]);
        }
      } else {
        rw[i] = zero8();
      }
    }
  };
  auto store_tile = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      *reinterpret_cast<half8_t*>(&lx[buf][xrow[i] * TL_LD + xcol[i]]) = rx[i];
      *reinterpret_cast<half8_t*>(&lw[buf][wrow[i] * TL_LD + wcol[i]]) = rw[i];
    }
  };

  float16_t acc[2][2];  // [tn][tm]
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.f;

  load_tile(0);
  store_tile(0);
  __syncthreads();
  for (int kt = 0; kt < nkt; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < nkt) load_tile(kt + 1);
#pragma unroll
    for (int ks = 0; ks < TL_BK / 16; ++ks) {
      half8_t fa[2], fb[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        fa[t] = *reinterpret_cast<const half8_t*>(
            &lw[buf][(wn * 64 + t * 32 + li) * TL_LD + ks * 16 + lg * 8]);
        fb[t] = *reinterpret_cast<const half8_t*>(
            &lx[buf][(wm * 64 + t * 32 + li) * TL_LD + ks * 16 + lg * 8]);
      }
#pragma unroll
      for (int tn = 0; tn < 2; ++tn)
#pragma unroll
        for (int tm = 0; tm < 2; ++tm)
          acc[tn][tm] = mfma_32x32x16<MODE>(fa[tn], fb[tm], acc[tn][tm]);
    }
    if (kt + 1 < nkt) store_tile(buf ^ 1);
    __syncthreads();
  }

  // MFMA 32x32 output: lane holds column (lane & 31) of B = activation row, and for register
  // v the A row 8*(v/4) + 4*(lane >> 5) + (v & 3) = output feature.
#pragma unroll
  for (int tn = 0; tn < 2; ++tn)
#pragma unroll
    for (int tm = 0; tm < 2; ++tm) {
      const int64_t m = m0 + wm * 64 + tm * 32 + li;
      if (m >= M) continue;
#pragma unroll
      for (int blk = 0; blk < 4; ++blk) {
        const int n = n0 + wn * 64 + tn * 32 + blk * 8 + lg * 4;
        if (n >= N) continue;
        const float4_t v = {acc[tn][tm][blk * 4 + 0], acc[tn][tm][blk * 4 + 1],
                            acc[tn][tm][blk * 4 + 2], acc[tn][tm][blk * 4 + 3]};
        epilogue4<MODE>(epi, m, n, v);
      }
    }
}

// ---- large tiled kernel, int8 weights --------------------------------------------------------
// 256 x 256 x 64 per workgroup of 8 waves on v_mfma_f32_16x16x32_f16; every wave owns 32 output
// features (two weight tiles) for all 256 activation rows.  Weight fragments come straight from
// the packed layout in global memory into registers (one KB per wave instruction, no LDS round
// trip, no two waves read the same weights); only the row-major activations are staged through
// LDS, double buffered, one barrier per 64-wide K stage.  A staged row is 128 bytes, unpadded, and
// its eight 16-byte chunks are stored XOR-swizzled by (row / 2) % 8: this part's LDS serves 256
// bytes per clock only when the 16 lanes it takes together hit 16 different 16-byte bank groups,
// which rows padded to 144 bytes do not (measured: 128 bytes per clock, i.e. the fragment reads of a
// stage alone took as long as its MFMAs).  The stage is software pipelined by
// hand: activations are fetched two stages ahead and parked in LDS one stage ahead, weights
// are fetched one stage ahead, LDS fragment reads run TB_PD fragments ahead of the MFMAs, and
// sched_group_barrier pins that order.  The main loop is branch free: rows and tiles past the
// edge read clamped addresses and are dropped in the epilogue.  Needs K % 128 == 0.
constexpr int TB_BM = 256, TB_BN = 256, TB_BK = 64, TB_LD = TB_BK, TB_THREADS = 512;
constexpr int TB_MF = TB_BM / 16;       // activation fragments per wave and 32-wide step
constexpr int TB_NT = TB_BN / 8 / 16;   // weight tiles per wave
constexpr int TB_PD = 4;                // LDS fragment reads in flight
constexpr int TB_LDS_BYTES = 2 * TB_BM * TB_LD * (int)sizeof(half_t);

struct BigW {  // one 64-wide stage of weights: 16 raw bytes per tile, the fragments of two steps
  half8_t f[TB_NT];
};

template <int MODE>
__global__ __launch_bounds__(TB_THREADS) void linear_tiled_big_kernel(
    const half_t* __restrict__ x, const void* __restrict__ Wp, const half_t* __restrict__ scales,
    int64_t M, int N, int K, Epilogue epi) {
  extern __shared__ __attribute__((aligned(16))) half_t lx_big[];  // [2][TB_BM * TB_LD]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lr = lane & 15, lg = lane >> 4;
  const int64_t m0 = (int64_t)blockIdx.y * TB_BM;
  const int n0 = blockIdx.x * TB_BN + wave * (TB_NT * 16);
  const int nkt = K / TB_BK;
  const int ntiles = N / 16;

  // activation staging: piece c = row c/8, 16-byte chunk c%8 (8 lanes cover one 128-byte line)
  const half_t* xsrc[4];
  int xdst[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = tid + TB_THREADS * i;
    const int row = c >> 3, ch = c & 7;
    const int64_t m = min(m0 + row, M - 1);
    xsrc[i] = x + m * K + ch * 8;
    xdst[i] = row * TB_LD + ((ch ^ ((row >> 1) & 7)) * 8);
  }
  const char* wsrc[TB_NT];
  half_t wscale[TB_NT];
#pragma unroll
  for (int j = 0; j < TB_NT; ++j) {
    const int t = min(n0 / 16 + j, ntiles - 1);
    wsrc[j] = (const char*)Wp + (int64_t)t * K * 16 + lane * 16;
    wscale[j] = scales[t * 16 + lr];
  }

  auto gload_x = [&](half8_t(&xr)[4], int kt) {
    kt = min(kt, nkt - 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) xr[i] = *reinterpret_cast<const half8_t*>(xsrc[i] + kt * TB_BK);
  };
  auto gload_w = [&](BigW& w, int kt) {
    kt = min(kt, nkt - 1);
#pragma unroll
    for (int j = 0; j < TB_NT; ++j) w.f[j] = *reinterpret_cast<const half8_t*>(wsrc[j] + (int64_t)kt * 1024);
  };
  auto lstore = [&](const half8_t(&xr)[4], int buf) {
    half_t* l = lx_big + buf * (TB_BM * TB_LD);
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<half8_t*>(l + xdst[i]) = xr[i];
  };

  float4_t acc[TB_MF][TB_NT];
#pragma unroll
  for (int a = 0; a < TB_MF; ++a)
#pragma unroll
    for (int b = 0; b < TB_NT; ++b) acc[a][b] = float4_t{0.f, 0.f, 0.f, 0.f};

  auto compute = [&](const BigW& w, int buf) {
    // fragment f = 32-wide step f / TB_MF, row block f % TB_MF: chunk 4 * step + lg of row
    // 16 * block + lr, whose swizzle is (lr / 2) % 8 for every block
    const half_t* lb = lx_big + buf * (TB_BM * TB_LD) + lr * TB_LD;
    const int sw = (lr >> 1) & 7;
    const half_t* l0 = lb + ((lg ^ sw) * 8);
    const half_t* l1 = lb + ((lg ^ sw ^ 4) * 8);
    auto frag = [&](int f) {
      return *reinterpret_cast<const half8_t*>((f / TB_MF ? l1 : l0) + (f % TB_MF) * 16 * TB_LD);
    };
    constexpr int F = 2 * TB_MF;
    half8_t a[2][TB_NT];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int j = 0; j < TB_NT; ++j) {
        const uint4 q = __builtin_bit_cast(uint4, w.f[j]);
        a[ks][j] = ks == 0 ? dequant8(q.x, q.y, wscale[j]) : dequant8(q.z, q.w, wscale[j]);
      }
    half8_t bx[TB_PD];
#pragma unroll
    for (int p = 0; p < TB_PD; ++p)
      bx[p] = frag(p);
    __builtin_amdgcn_sched_group_barrier(0x200, 4, 0);          // LDS stores
    __builtin_amdgcn_sched_group_barrier(0x020, 4 + TB_NT, 0);  // global loads
    __builtin_amdgcn_sched_group_barrier(0x100, TB_PD, 0);      // leading LDS reads
#pragma unroll
    for (int f = 0; f < F; ++f) {
      const int ks = f / TB_MF, mf = f % TB_MF;
      const half8_t cur = bx[f % TB_PD];
#pragma unroll
      for (int j = 0; j < TB_NT; ++j)
        acc[mf][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[ks][j], cur, acc[mf][j], 0, 0, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, TB_NT, 0);
      if (f + TB_PD < F) {
        bx[f % TB_PD] = frag(f + TB_PD);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
    }
  };

  half8_t xr[4];
  BigW w0, w1;
  gload_x(xr, 0);
  gload_w(w0, 0);
  lstore(xr, 0);
  gload_x(xr, 1);
  __syncthreads();
  for (int kt = 0; kt < nkt; kt += 2) {
    lstore(xr, 1);  // stage kt + 1, fetched during stage kt - 1
    gload_x(xr, kt + 2);
    gload_w(w1, kt + 1);
    compute(w0, 0);
    __syncthreads();
    lstore(xr, 0);
    gload_x(xr, kt + 3);
    gload_w(w0, kt + 2);
    compute(w1, 1);
    __syncthreads();
  }

  // D of the 16x16 MFMA: lane holds activation row (lane & 15) and the 4 consecutive features
  // 4 * (lane >> 4) .. + 3 of the weight tile
#pragma unroll
  for (int mf = 0; mf < TB_MF; ++mf) {
    const int64_t m = m0 + mf * 16 + lr;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < TB_NT; ++j) {
      const int n = n0 + j * 16;
      if (n >= N) continue;
      epilogue4<MODE>(epi, m, n + lg * 4, acc[mf][j]);
    }
  }
}

// ---- large tiled kernel, fp16 weights: four waves of 128 x 128 ---------------------------------
// 256 x 256 per workgroup of 4 waves (2 x 2), one wave per SIMD, each wave 128 rows x 128 features
// on v_mfma_f32_16x16x32_f16: 64 accumulator tiles = 256 registers, kept in the AGPR bank.  hipcc
// copies such accumulators in and out of the bank around every MFMA, so the MFMAs are issued from
// inline assembly with the accumulator tied in place ("+a").  Both operands go global -> LDS
// directly (global_load_lds_dwordx4: LDS address = M0 + instruction offset + 16 * lane, global
// address = scalar base + lane offset + the same instruction offset), so no load ever targets a
// register and the only hand-placed waits are the vmcnt before each barrier:
//   * activations in 64-wide stages (whole 128-byte lines), rows unpadded with their eight 16-byte
//     chunks XOR-swizzled by (row / 2) % 8, ring of 3 x 32 KB (256 rows);
//   * weights in 32-wide steps, the packed 16 x 32 blocks as they lie in memory (lane order, so the
//     fragment reads are linear), ring of 4 x 16 KB (256 columns).
// A group of loads (the RF of a wave's share of a stage, the WF / 2 of its share of a step) shares one
// M0 and one lane offset; the instruction offset picks the 1 KB piece, and the scalar bases, which
// are loop invariant, are moved back by it.
// One barrier per 32-wide step.  Behind the barrier of step t the weights of step t+1 (and, every
// other step, the activations of the next stage) are complete and the buffers of step t are free:
// the loads of step t+4 / stage S+2 are issued there, one between every few MFMAs, and the 16
// fragments of step t+1 are read under the 64 MFMAs of step t (one ds_read_b128 per 4 MFMAs, a
// quarter of the LDS traffic per MFMA of the 8-wave kernel above).
// Epilogue through LDS: a lane holds 4 features of 16 different rows per tile, which as stores are
// 32-byte pieces; the rounded tile rows are parked in LDS and read back as 16 bytes per lane, whole
// 256-byte row pieces per 16 lanes.
// Workgroup -> tile: consecutive workgroups land on consecutive XCDs; where the default order would
// give an XCD a long thin strip of a round's tiles, the 256 tiles of a round are regrouped so that
// every XCD's L2 serves a compact a x b block (rm_a, rm_r from the host; rm_a < 0: by panels).
// Three widths of the workgroup's tile, by the number WF of 16-feature weight fragments per wave:
// 8 -> 256 x 256 (as described), 4 -> 256 x 128, 2 -> 256 x 64 (fewer accumulators, weight loads and
// MFMAs per step; the same activation stages).  The two wider forms need M >= 256: a ragged last
// row tile is moved up to end at M and stores only the rows no other tile owns.  The narrowest
// form repeats the last row in its loads instead and drops the rows past it, so it also serves
// fewer than 256 rows, as does any form with FEW.  RF = 4 .. 8 16-row activation fragments per wave: tiles of 32 RF
// rows, whose rings are as deep as the LDS allows (128 x 128: five stages and eight steps).  All need K % 64 == 0, K >= 128.
constexpr int TQ_BM = 256, TQ_THREADS = 256;  // (rows of a tile unless RF is given)
constexpr int TQ_PANEL = 16;  // columns of tiles taken together where many lie across
constexpr int tq_bm(int RF) { return 32 * RF; }
// stages of activations and steps of weights in the rings: as many as 160 KB hold, steps for all but one stage
constexpr int tq_rx(int RF, int WF) { return RF == 4 && WF == 4 ? 5 : RF == 4 || (RF < 8 && WF == 4) ? 4 : 3; }
constexpr int tq_rw(int RF, int WF) { return 2 * (tq_rx(RF, WF) - 1); }
constexpr int tq_xbytes(int RF) { return tq_bm(RF) * 64 * 2; }  // one 64-wide stage of activations
constexpr int tq_bn(int WF) { return 32 * WF; }
constexpr int tq_wbytes(int WF) { return 2 * WF * 1024; }  // one 32-wide step of weights
// KB of columns x rows: 256 x 256 160, x 224 148, x 192 136, x 160 124, x 128 160; 128 x 256 128, x 224 160, x 192 144, x 160
// 128, x 128 144; 64 x 256 112
constexpr int tq_lds_bytes(int WF, int RF = 8) {
  return tq_rx(RF, WF) * tq_xbytes(RF) + tq_rw(RF, WF) * tq_wbytes(WF);
}
constexpr bool tq_lds_fits(int WF, int lo) {
  for (int rf = lo; rf <= 8; ++rf)
    if (tq_lds_bytes(WF, rf) > 160 * 1024) return false;
  return true;
}
static_assert(tq_lds_fits(8, 4) && tq_lds_fits(4, 4) && tq_lds_fits(2, 8), "a CU has 160 KB of LDS");
typedef __attribute__((address_space(3))) void tq_lds_void;

template <int MODE>
__device__ __forceinline__ void tq_mfma(float4_t& acc, const half8_t& a, const half8_t& b) {
  if constexpr (is_bf<MODE>)
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
  else
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}

// Which of a step's RF x WF MFMAs (row * WF + column) is the q-th: two rows side by side, column after column, back and
// forth.  What an MFMA draws depends on the operands of the one before it, and the part lowers its clock by that:
// MFMAs alone, random operands, 1.91 PFLOP/s row by row, 1.96 so (one operand new each time, a snake of rows, 1.93;
// both new 1.84; four rows side by side 1.90).  32768 x 16384 x 4096 3118 -> 3075 us, 2048 x 16384 x 4096 206 -> 200.
// Not of 64 columns: those tiles draw less, and a step of 16 MFMAs waits for two rows of fragments in front of its first
// pair (row by row and so, us: bf16 147 x 416 x 7104 50.2 and 54.1, 182 x 288 x 2944 14.2 and 14.8, fp16 83 x 7168 x 28672 in two
// slices 133 and 137).
constexpr int tq_order(int RF, int WF, int q) {
  if (WF == 2) return q;
  const int g = q / (2 * WF), w = q % (2 * WF);
  if (2 * g + 1 >= RF) return 2 * g * WF + (g & 1 ? WF - 1 - w : w);
  const int c = w / 2;
  return (2 * g + (w & 1)) * WF + (g & 1 ? WF - 1 - c : c);
}

template <int... I, class F>
__device__ __forceinline__ void tq_static_for_impl(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void tq_static_for(F&& f) {
  tq_static_for_impl(std::make_integer_sequence<int, N>{}, f);
}

// 8 consecutive output columns n..n+7 of row m; v holds the accumulators rounded to fp16, b the
// bias and r the residual values of those columns (read only where the epilogue has them)
__device__ __forceinline__ void biased8(const Epilogue& e, half8_t v, half8_t b, float (&t)[8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) t[i] = (float)v[i];
  if (e.bias) {
#pragma unroll
    for (int i = 0; i < 8; ++i) t[i] = round_h(t[i] + (float)b[i]);
  }
}
__device__ __forceinline__ void epilogue8(const Epilogue& e, int64_t m, int n, half8_t v, half8_t b, half8_t r) {
  float t[8];
  biased8(e, v, b, t);
  half8_t o;
  if (e.flags & MSA_EPI_RELU) {
#pragma unroll
    for (int i = 0; i < 8; ++i) t[i] = fmaxf(t[i], 0.f);
  }
  if (e.residual) {
#pragma unroll
    for (int i = 0; i < 8; ++i) t[i] = round_h(t[i] + (float)r[i]);
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = (half_t)t[i];
  if (e.out_mb > 0)
    *reinterpret_cast<half8_t*>(e.y + packed_act_offset((int)m, n, e.out_mb)) = o;
  else
    *reinterpret_cast<half8_t*>(e.y + m * e.N + n) = o;
}

// Row tiles of a grouped product (routed experts): tile t holds rows tile_row[t] .. of group
// tile_group[t], at most TQ_BM of them and none past group_end; row r of the product reads row
// perm[r] / rows_per_x of the activations (perm NULL: row r) and multiplies the group's own matrix.
struct GroupTiles {
  const int32_t *perm, *tile_group, *tile_row, *n_tiles, *group_end;
  int rows_per_x;
};

// GROUPED: the row tiles come from `gt`; every XCD takes a contiguous share of the tiles, columns
// fastest, so that the column tiles of a row tile run side by side behind one L2.
// PART: split-K.  Workgroup (bx, by, z) sums over the K range of ``part_stages`` 64-wide stages
// that starts at stage z * part_stages and stores its fp32 sums, with no epilogue, as slice z of
// ``part`` ([gridDim.z][M][N]); a later launch adds the slices in slice order.
// m_own: the first row that the tile owns.
// ONCE: one row of tiles (or an expert's only one), so that a weight is read by one workgroup: its loads leave nothing in
// the caches and are served faster (us: 200 x 50272 x 4096 101 -> 96, 100 x 50272 x 4096 84 -> 73, 70 x 16384 x 4096 43.9 -> 41.8;
// two rows of tiles would lose by it, 129 x 12288 x 4096 33.3 -> 39.3).  Sums in slices are not: by themselves they gain, 146 rows
// of 8192 x 4608 27.4 -> 26.7, but not with the tail that reads them, 32.5 -> 34.4; bf16, 156 x 4096 x 3072 17.8 -> 19.9, 200 x
// 4096 x 4096 22.0 -> 22.2; 4096 x 16384 of 130, 200 and 250 rows 44.1 -> 45.1, 46.3 -> 45.7, 49.3 -> 48.0.
template <int MODE, int WF, bool PART, bool GROUPED, int RF, bool FEW, bool ONCE = false>
__device__ __forceinline__ void quad_tile(const half_t* __restrict__ x, const void* __restrict__ Wp, int64_t M, int N,
                                          int K, int bx, int64_t m_own, int bz, const Epilogue& epi,
                                          float* __restrict__ part, int part_stages, const GroupTiles& gt) {
  extern __shared__ __attribute__((aligned(16))) char tq_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int wm = wave >> 1, wn = wave & 1;
  constexpr int TQ_BN = tq_bn(WF), TQ_WBYTES = tq_wbytes(WF), TQ_BM = tq_bm(RF), TQ_XBYTES = tq_xbytes(RF);
  constexpr int TQ_RX = tq_rx(RF, WF), TQ_RW = tq_rw(RF, WF), TQ_WOFF = TQ_RX * TQ_XBYTES;
  constexpr int WL = WF / 2;  // weight load instructions per wave and step
  constexpr int XL = RF;      // activation load instructions per wave and stage
  // The narrowest form (WF = 2) also serves fewer than 256 rows: it does not move a ragged tile up
  // but repeats the last row in its loads and drops the rows past it in the epilogue.  So does
  // the split-K form of WF = 4 (decode batches of 129 .. 255 rows cut K eight ways over it).
  constexpr bool CLAMP = WF == 2 || (WF == 4 && PART) || GROUPED || (RF == 4 && WF == 4) || FEW;
  const int64_t m0 = !CLAMP && m_own + TQ_BM > M ? M - TQ_BM : m_own;
  const int n0 = bx * TQ_BN;
  // the stages this workgroup sums over: all of K, or its slice (the operand bases below move
  // to the slice's first stage, so that stage and step numbers count from 0 either way)
  const int st_first = PART ? bz * part_stages : 0;
  const int nst = PART ? part_stages : K / 64, nks = 2 * nst;
  const int ntiles = N / 16;

  // direct loads.  Activations, per stage: instruction i (0 .. RF - 1) of the wave fills rows
  // 8 RF * wave + 8 * i .. + 7 (lane l: row l / 8, chunk position l % 8, which must hold chunk
  // (l % 8) ^ ((row / 2) % 8) = (l % 8) ^ (4 * (i % 2) + l / 16), or 4 * ((i + 1) % 2) where RF * wave is
  // odd), with M0 at the wave's piece + RF / 2 KB and instruction offset 1024 * (i - RF / 2).  Weights, per
  // step: the wave copies the blocks of tiles WL * wave .. WL * wave + WL - 1, instruction offset 1024 * j.
  const char* xb[XL];
  const char* wb[WL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int64_t r = m0 + wave * (TQ_BM / 4) + i * 8;
    const int64_t base_row = GROUPED ? 0 : CLAMP ? min(r, M - 1) : r;
    xb[i] = (const char*)(x + base_row * K + (int64_t)st_first * 64) - (i - XL / 2) * 1024;
  }
#pragma unroll
  for (int j = 0; j < WL; ++j) {
    const int tt = min(n0 / 16 + wave * WL + j, ntiles - 1);
    wb[j] = (const char*)Wp + (int64_t)tt * K * 32 + (int64_t)st_first * 2048 - j * 1024;
  }
  const uint32_t xrow = (uint32_t)(lane >> 3) * (uint32_t)K * 2;
  const uint32_t xlane0 = xrow + (((lane & 7) ^ (lane >> 4)) * 16);
  const uint32_t xlane1 = xrow + (((lane & 7) ^ (4 + (lane >> 4))) * 16);
  // (an odd RF: the second and the fourth wave's rows begin at an odd multiple of eight)
  const bool swap = RF % 2 && (wave & 1);
  const uint32_t xeven = swap ? xlane1 : xlane0, xodd = swap ? xlane0 : xlane1;
  const uint32_t wlane = lane * 16;
  // CLAMP: per instruction, the lane's row offset from the (clamped) scalar base row
  uint32_t xl[CLAMP ? XL : 1];
  if (CLAMP) {
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int64_t r = m0 + wave * (TQ_BM / 4) + i * 8;
      int64_t d = min(r + (lane >> 3), M - 1);
      if (GROUPED) {
        if (gt.perm) d = gt.perm[d] / gt.rows_per_x;
      } else {
        d -= min(r, M - 1);
      }
      xl[i] = (uint32_t)d * (uint32_t)K * 2 + ((i & 1 ? xodd : xeven) - xrow);
    }
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(tq_lds_void*)tq_lds;
  // Lane offsets and LDS base of the group being issued.  The LDS base travels in M0, which every
  // load names as an explicit register operand: the compiler then knows that M0 is live between
  // the loads of a group (ordinary code - fragment reads, MFMAs - runs between them) and writes
  // it once per group.
  uint32_t xv0 = 0, xv1 = 0, wv = 0, xst = 0, xm0 = 0, wm0 = 0;
  auto set_x = [&](int slot, int st) {
    st = min(st, nst - 1);
    xst = st * 128;
    xv0 = xeven + st * 128;
    xv1 = xodd + st * 128;
    xm0 = lds0 + slot * TQ_XBYTES + wave * (TQ_BM / 4 * 128) + XL / 2 * 1024;
  };
  auto set_w = [&](int slot, int ks) {
    ks = min(ks, nks - 1);
    wv = wlane + ks * 1024;
    wm0 = lds0 + TQ_WOFF + slot * TQ_WBYTES + wave * (WL * 1024);
  };
  auto issue_x = [&](auto ic) {
    constexpr int i = decltype(ic)::value;
    const uint32_t vo = CLAMP ? xl[CLAMP ? i : 0] + xst : (i & 1 ? xv1 : xv0);
    const char* sb = xb[i];
    const uint32_t base = xm0;
    asm volatile("global_load_lds_dwordx4 %0, %1 offset:%2" ::"v"(vo), "s"(sb),
                 "n"((i - XL / 2) * 1024), "{m0}"(base)
                 : "memory");
  };
  auto issue_w = [&](auto jc) {
    constexpr int j = decltype(jc)::value;
    const uint32_t vo = wv;
    const char* sb = wb[j];
    const uint32_t base = wm0;
    if constexpr (ONCE)
      asm volatile("global_load_lds_dwordx4 %0, %1 offset:%2 nt" ::"v"(vo), "s"(sb), "n"(j * 1024),
                   "{m0}"(base)
                   : "memory");
    else
      asm volatile("global_load_lds_dwordx4 %0, %1 offset:%2" ::"v"(vo), "s"(sb), "n"(j * 1024),
                   "{m0}"(base)
                   : "memory");
  };
  auto group_x = [&](int slot, int st) {
    set_x(slot, st);
    tq_static_for<XL>([&](auto ic) { issue_x(ic); });
  };
  auto group_w = [&](int slot, int ks) {
    set_w(slot, ks);
    tq_static_for<WL>([&](auto jc) { issue_w(jc); });
  };

  // fragment reads.  Activation fragment i of half h of a stage: row 16 RF * wm + 16 * i + lr, chunk
  // 4 * h + lg at position (4 * h + lg) ^ ((lr / 2) % 8); weight fragment j: tile WF * wn + j.
  const int sw = (lr >> 1) & 7;
  const uint32_t xoff0 = (uint32_t)(wm * (TQ_BM / 2) + lr) * 128 + ((lg ^ sw) * 16);
  const uint32_t xoff1 = (uint32_t)(wm * (TQ_BM / 2) + lr) * 128 + ((lg ^ sw ^ 4) * 16);
  const uint32_t woff = TQ_WOFF + (uint32_t)(wn * WF) * 1024 + lane * 16;
  auto xfrag = [&](int slot, int h, int i) {
    return *reinterpret_cast<const half8_t*>(tq_lds + slot * TQ_XBYTES + (h ? xoff1 : xoff0) +
                                             i * (16 * 128));
  };
  auto wfrag = [&](int slot, int j) {
    return *reinterpret_cast<const half8_t*>(tq_lds + slot * TQ_WBYTES + woff + j * 1024);
  };

  float4_t acc[RF][WF];
#pragma unroll
  for (int i = 0; i < RF; ++i)
#pragma unroll
    for (int j = 0; j < WF; ++j) {
      acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
      asm volatile("" : "+a"(acc[i][j]));
    }

  // prologue.  A ring of three stages: activation stages 0 and 1, weight steps 0..3 requested; stages 0, 1 and steps 0,
  // 1 landed
  half8_t xf[2][RF], wf[2][WF];
  if constexpr (TQ_RX == 3) {
    group_x(0, 0);
    group_w(0, 0);
    group_x(1, 1);
    group_w(1, 1);
    group_w(2, 2);
    group_w(3, 3);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * WL) : "memory");
  } else {  // as the steps -TQ_RW .. -1 would have requested them; stage 0 and step 0 landed
#pragma unroll
    for (int v = 0; v < TQ_RW; ++v) {
      if (v % 2 == 0) group_x(v / 2, v / 2);
      group_w(v, v);
    }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(TQ_RW / 2 * XL + TQ_RW * WL - XL - WL) : "memory");
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < RF; ++i) xf[0][i] = xfrag(0, 0, i);
#pragma unroll
  for (int j = 0; j < WF; ++j) wf[0][j] = wfrag(0, j);

  // step t = 2 S + H; xs, ws: ring slots of stage S and step t.  An even step issues RF + WL loads
  // (stage S + TQ_RX - 1, then step t + TQ_RW), an odd one WL (step t + TQ_RW).  Loads complete in order; the weights
  // of step t + 1 were requested TQ_RW - 1 steps ago, and the loads of the TQ_RW - 2 steps since may still be
  // outstanding at the barrier, half of them with activations.  The activations an odd step starts to read
  // (stage S + 1) were requested in the same step as its weights, ahead of them.
  // The RF x WF MFMAs of a step carry, one each: the RF + WF fragment reads of step t + 1 and the
  // loads (RF = 8, even steps: activations under rows 0..3, weights under rows 4..7).
  auto step = [&](int t, int xs, int ws, auto hc) {
    constexpr int H = decltype(hc)::value;
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((TQ_RW - 2) / 2 * XL + (TQ_RW - 2) * WL) : "memory");
    __syncthreads();
    const int S = t >> 1;
    const int xfree = xs == 0 ? TQ_RX - 1 : xs - 1;  // slot of stage S - 1 = slot of stage S + TQ_RX - 1
    const int xnext = xs == TQ_RX - 1 ? 0 : xs + 1;  // slot of stage S + 1
    const int wnext = ws == TQ_RW - 1 ? 0 : ws + 1;  // slot of step t + 1
    tq_static_for<RF>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      tq_static_for<WF>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        constexpr int o = tq_order(RF, WF, i * WF + j);
        tq_mfma<MODE>(acc[o / WF][o % WF], wf[H][o % WF], xf[H][o / WF]);
        if constexpr (RF < 8 && !(RF == 4 && WF == 4)) {
          // one instruction behind an MFMA: fragments of step t + 1, then a row's load of activations (even steps)
          // and one of weights
          if (j == 1) xf[H ^ 1][i] = H == 0 ? xfrag(xs, 1, i) : xfrag(xnext, 0, i);
          if constexpr (WF == 8) {
            if constexpr (j == 5) wf[H ^ 1][i] = wfrag(wnext, i);
            if constexpr (j == 7 && RF + i < WF) wf[H ^ 1][(RF + i) % WF] = wfrag(wnext, (RF + i) % WF);
          } else {
            if constexpr (j == 3 && i < WF) wf[H ^ 1][i % WF] = wfrag(wnext, i % WF);
          }
          if constexpr (H == 0) {
            if (i == 0 && j == 0) set_x(xfree, S + TQ_RX - 1);
            if constexpr (j == 0) issue_x(ic);
          }
          if (i == 0 && j == 1) set_w(ws, t + TQ_RW);
          if constexpr (WF == 8) {
            if constexpr (j == 3 && i < WL) issue_w(std::integral_constant<int, i % WL>{});
          } else {
            if constexpr (j == 2 && (i == 1 || i == 3)) issue_w(std::integral_constant<int, (i >> 1) % WL>{});
          }
        } else if constexpr (RF == 4) {
          if (j == 1) xf[H ^ 1][i] = H == 0 ? xfrag(xs, 1, i) : xfrag(xnext, 0, i);
          if (j == 3) wf[H ^ 1][i] = wfrag(wnext, i);
          if constexpr (H == 0) {
            if (i == 0 && j == 0) set_x(xfree, S + TQ_RX - 1);
            if (j == 0) issue_x(ic);
          }
          if (i == 0 && j == 1) set_w(ws, t + TQ_RW);
          if constexpr (j == 2 && (i & 1)) issue_w(std::integral_constant<int, (i >> 1)>{});
        } else {
          if (j == 1) xf[H ^ 1][i] = H == 0 ? xfrag(xs, 1, i) : xfrag(xnext, 0, i);
          if constexpr (WF == 8) {
            if (j == 5) wf[H ^ 1][i % WF] = wfrag(wnext, i % WF);
          } else if constexpr (WF == 4) {
            if constexpr (j == 3 && (i & 1)) wf[H ^ 1][(i >> 1) % WF] = wfrag(wnext, (i >> 1) % WF);
          } else {
            if constexpr (j == 0 && (i == 1 || i == 5)) wf[H ^ 1][(i >> 2) % WF] = wfrag(wnext, (i >> 2) % WF);
          }
          if constexpr (H == 0) {
            if (i == 0 && j == 0) set_x(xfree, S + 2);
            if constexpr (i < 4 && j == WF / 2 - 1) issue_x(std::integral_constant<int, (i & 3) * 2>{});
            if constexpr (i < 4 && j == WF - 1) issue_x(std::integral_constant<int, (i & 3) * 2 + 1>{});
            if (i == 4 && j == 0) set_w(ws, t + TQ_RW);
            if constexpr (WF == 8) {
              if constexpr (i >= 4 && j == 3) issue_w(std::integral_constant<int, (i & 3) % WL>{});
            } else if constexpr (WF == 4) {
              if constexpr ((i == 4 || i == 6) && j == 2)
                issue_w(std::integral_constant<int, ((i >> 1) & 1) % WL>{});
            } else {
              if constexpr (i == 4 && j == 1) issue_w(std::integral_constant<int, 0>{});
            }
          } else {
            if (i == 0 && j == 0) set_w(ws, t + TQ_RW);
            if constexpr (WF == 8) {
              if constexpr (j == 3 && (i & 1)) issue_w(std::integral_constant<int, (i >> 1) % WL>{});
            } else if constexpr (WF == 4) {
              if constexpr ((i == 2 || i == 6) && j == 2)
                issue_w(std::integral_constant<int, ((i >> 2) & 1) % WL>{});
            } else {
              if constexpr (i == 2 && j == 1) issue_w(std::integral_constant<int, 0>{});
            }
          }
        }
      });
    });
  };
  int xs = 0, ws = 0;
  // Where the loop begins shows: with one wave per SIMD its fetches have nothing beside them.  The wider forms begin at
  // (or 4 bytes past) a 128-byte line of instructions (1500 x 3072 x 4096 on 256 x 128 tiles 51 us, 60 bytes past
  // a line 52.6; 2005 x 4096 x 16384 224 us, 32 past 230), the narrowest 32 or 36 bytes past one (200 x 2048
  // x 1024 12.5 us, at a line or 24 past 12.9).  The fills leave room for the few scalar instructions that the
  // compiler puts behind them.
  asm volatile(".p2align 7\n\t.fill %3, 4, 0xbf800000" ::"s"(nks), "s"(xs), "s"(ws), "n"(WF > 2 ? 25 : 2) : "memory");
  for (int t = 0; t < nks; t += 2) {
    step(t, xs, ws, std::integral_constant<int, 0>{});
    ws = ws == TQ_RW - 1 ? 0 : ws + 1;
    step(t + 1, xs, ws, std::integral_constant<int, 1>{});
    ws = ws == TQ_RW - 1 ? 0 : ws + 1;
    xs = xs == TQ_RX - 1 ? 0 : xs + 1;
  }
  // no direct load may still be in flight when the rings are reused below (or when the workgroup's
  // LDS is released); the last MFMAs must have written their accumulators before these are read
  // (the compiler does not see MFMAs inside the asm)
  asm volatile("s_waitcnt vmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");
  // ties every accumulator to this point: none of their reads may be scheduled above the wait
#pragma unroll
  for (int i = 0; i < RF; ++i)
#pragma unroll
    for (int j = 0; j < WF; ++j) asm volatile("" : "+a"(acc[i][j]));
  __syncthreads();  // every wave is done with the operand rings

  if constexpr (PART) {
    // the sums as the lanes hold them: D tile (i, j) = activation row 16 * i + lr of the wave's
    // 128, features 16 * j + 4 * lg .. + 3 of the wave's 16 WF (16 bytes per lane, 64 per row)
    float* slice = part + (int64_t)bz * M * N;
#pragma unroll
    for (int i = 0; i < RF; ++i) {
      const int64_t m = m0 + wm * (TQ_BM / 2) + i * 16 + lr;
#pragma unroll
      for (int j = 0; j < WF; ++j) {
        const int n = n0 + wn * (16 * WF) + 16 * j + 4 * lg;
        if (m >= m_own && m < M && n < N)
          *reinterpret_cast<float4_t*>(slice + m * N + n) = acc[i][j];
      }
    }
    return;
  }

  if constexpr (is_bf<MODE>) {
    // As below, through LDS so that whole row pieces are stored; the GLU form halves the columns
    // (two outputs per lane and tile).  Tiles from column n32 on leave as the lanes hold them.
    constexpr bool GLU = MODE == MODE_BF_GLU;
    constexpr int BCH = GLU ? WF : 2 * WF;  // 16-byte chunks of a staged row
    constexpr int BRB = 16 * BCH;           // bytes of a staged row
    constexpr int BRPI = 64 / BCH;          // rows a 64-lane read covers
    constexpr int BNR = (16 + BRPI - 1) / BRPI;
    char* stage = tq_lds + wave * 8192;
    const int bc = lane % BCH, brow = lane / BCH;
    const int nw = n0 + wn * (16 * WF);      // first column of the wave
    const int bn = GLU ? (nw >> 1) + bc * 8 : nw + bc * 8;  // first output column of the lane
    const bool bn_ok = bn < (GLU ? epi.n32 >> 1 : epi.n32);
    // (read once: behind the first store the compiler may no longer keep them)
    PostVectors post[MODE == MODE_BF_POST ? WF : 1];
    if constexpr (MODE == MODE_BF_POST) {
#pragma unroll
      for (int j = 0; j < WF; ++j) post[j] = post_vectors(epi, min(nw + 16 * j, N - 16) + 4 * lg);
    }
#pragma unroll
    for (int i = 0; i < RF; ++i) {
      char* buf = stage + (i & 1) * 4096;
      const int64_t mf = m0 + wm * (TQ_BM / 2) + i * 16 + lr;
#pragma unroll
      for (int j = 0; j < WF; ++j) {
        const int n = nw + 16 * j + 4 * lg;
        if constexpr (MODE == MODE_BF_POST) acc[i][j] = post4(epi, nw + 16 * j, acc[i][j], post[j]);
        if (nw + 16 * j >= epi.n32) {  // wave-uniform: n32 is a multiple of 16
          if (mf >= m_own && mf < M && n < N)
            *reinterpret_cast<float4_t*>(epi.y32 + mf * (N - epi.n32) + (n - epi.n32)) = acc[i][j];
        } else if constexpr (GLU) {
          const bf16x2_t o = {(bf16_t)glu_act(epi.glu, acc[i][j][0], acc[i][j][1], epi.limit),
                              (bf16_t)glu_act(epi.glu, acc[i][j][2], acc[i][j][3], epi.limit)};
          *reinterpret_cast<bf16x2_t*>(buf + lr * BRB + ((j ^ (lr & (BCH - 1))) * 16) + lg * 4) = o;
        } else {
          const bf16x4_t o = {(bf16_t)acc[i][j][0], (bf16_t)acc[i][j][1], (bf16_t)acc[i][j][2],
                              (bf16_t)acc[i][j][3]};
          const int c = (2 * j + (lg >> 1)) ^ (lr & (BCH - 1));
          *reinterpret_cast<bf16x4_t*>(buf + lr * BRB + c * 16 + (lg & 1) * 8) = o;
        }
      }
#pragma unroll
      for (int r = 0; r < BNR; ++r) {
        const int row = BRPI * r + brow;
        if (row >= 16) continue;
        const half8_t v = *reinterpret_cast<const half8_t*>(buf + row * BRB +
                                                            ((bc ^ (row & (BCH - 1))) * 16));
        const int64_t m = m0 + wm * (TQ_BM / 2) + i * 16 + row;
        bf16_t* y = epi.yb + m * epi.ldy + bn;
        if constexpr (MODE == MODE_BF_POST)
          if (bn >= epi.n2) y = epi.y2 + m * epi.ld2 + (bn - epi.n2);
        if (bn_ok && m >= m_own && m < M) *reinterpret_cast<half8_t*>(y) = v;
      }
    }
    return;
  }

  // D tile (i, j): the lane holds activation row 16 * i + lr of the wave's 128 and the 4 features
  // 16 * j + 4 * lg ...  Per i the wave's 16 rows x 16 WF features (4 or 2 KB, two buffers per wave)
  // are written as the lanes hold them (16-byte chunk 2 j + lg / 2 of the row, swizzled by the row)
  // and read back 16 bytes per lane, whole rows per 16 (8) lanes.
  // The lane's column group is the same in every iteration, so the bias is read once; the residual
  // rows are requested four iterations ahead (the fragment registers are free now), so that their
  // latency is paid once per workgroup and not once per iteration.
  char* mine = tq_lds + wave * 8192;
  constexpr int ECH = 2 * WF;        // 16-byte chunks of a staged row (16 WF features)
  constexpr int ERB = 16 * ECH;      // bytes of a staged row
  constexpr int ERPI = 64 / ECH;     // rows a 64-lane read covers
  constexpr int ENR = 16 / ERPI;     // reads per 16 rows
  const int ec = lane % ECH, erow = lane / ECH;
  const int en = n0 + wn * (16 * WF) + ec * 8;
  const bool col_ok = en < N;
  half8_t bias8 = zero8();
  if (epi.bias && col_ok) bias8 = *reinterpret_cast<const half8_t*>(epi.bias + en);
  constexpr int TQ_RES_AHEAD = 4;
  half8_t res8[TQ_RES_AHEAD][ENR];
  auto load_res = [&](int i, half8_t(&dst)[ENR]) {
    if (MODE != MODE_PLAIN || !epi.residual) return;
#pragma unroll
    for (int r = 0; r < ENR; ++r) {
      const int64_t m = m0 + wm * (TQ_BM / 2) + i * 16 + ERPI * r + erow;
      if (col_ok && m >= m_own && m < M)
        dst[r] = *reinterpret_cast<const half8_t*>(epi.residual + m * epi.N + en);
    }
  };
#pragma unroll
  for (int i = 0; i < TQ_RES_AHEAD; ++i) load_res(i, res8[i]);
  // QKV mode: where a row's keys and values go (elements in front of its first head's, -1: nowhere) is worked out
  // once per row, two rows to a lane, and kept in LDS; the lane's columns are the same in every iteration, so their part
  // and head are constants.  (Kept in registers instead, positions, cache rows and divisions spilled 196 of
  // them: 1607 x 12288 x 4096 into cache rows of their own 179 us, now 156, as the plain product; 3000 rows 277 and 243.)
  const int64_t* place = reinterpret_cast<const int64_t*>(tq_lds + 32768 + wave * (TQ_BM / 2 * 8));
  half_t* to = nullptr;
  int qkv_part = 0;
  if constexpr (MODE == MODE_QKV) {
    int64_t* fill = reinterpret_cast<int64_t*>(tq_lds + 32768 + wave * (TQ_BM / 2 * 8));
#pragma unroll
    for (int k = 0; k < TQ_BM / 2; k += 64) {
      const int m = (int)min(m0 + wm * (TQ_BM / 2) + k + lane, M - 1);
      int b = m, at = epi.S0;
      bool ok = epi.S0 >= 0;
      if (epi.len_dev) {
        at = epi.len_dev[m];
        if (epi.row_dev) b = epi.row_dev[m];
        ok = at >= 0;
      } else if (epi.T > 1) {
        b = m / epi.T;
        at += m - b * epi.T;
      }
      if (TQ_BM / 2 % 64 == 0 || k + lane < TQ_BM / 2)
        fill[k + lane] = ok && at < epi.S_cap ? ((int64_t)b * epi.H * epi.S_cap + at) * epi.hd : -1;
    }
    const int D = epi.H * epi.hd;
    qkv_part = (en >= D) + (en >= 2 * D);  // 0 = K, 1 = V, 2 = Q
    const int c = en - qkv_part * D, h = epi.hd_shift >= 0 ? c >> epi.hd_shift : c / epi.hd;
    to = qkv_part == 2 ? epi.q_out + c
                       : (qkv_part == 0 ? epi.Kc : epi.Vc) + (int64_t)h * epi.S_cap * epi.hd + (c - h * epi.hd);
  }
#pragma unroll
  for (int i = 0; i < RF; ++i) {
    char* buf = mine + (i & 1) * 4096;
#pragma unroll
    for (int j = 0; j < WF; ++j) {
      half4_t o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (half_t)(acc[i][j][e]);
      const int c = (2 * j + (lg >> 1)) ^ (lr & (ECH - 1));
      *reinterpret_cast<half4_t*>(buf + lr * ERB + c * 16 + (lg & 1) * 8) = o;
    }
#pragma unroll
    for (int r = 0; r < ENR; ++r) {
      const int row = ERPI * r + erow;
      const half8_t v = *reinterpret_cast<const half8_t*>(buf + row * ERB +
                                                          ((ec ^ (row & (ECH - 1))) * 16));
      const int64_t m = m0 + wm * (TQ_BM / 2) + i * 16 + row;
      if (col_ok && m >= m_own && m < M) {
        if constexpr (MODE == MODE_QKV) {
          const int64_t at = qkv_part == 2 ? m * (epi.H * epi.hd) : place[i * 16 + row];
          if (at >= 0) {
            float t[8];
            biased8(epi, v, bias8, t);
            half8_t o;
            const float scale = qkv_part == 2 ? epi.qscale : 1.f;
#pragma unroll
            for (int k = 0; k < 8; ++k) o[k] = (half_t)(t[k] * scale);
            *reinterpret_cast<half8_t*>(to + at) = o;
          }
        } else {
          epilogue8(epi, m, en, v, bias8, res8[i % TQ_RES_AHEAD][r]);
        }
      }
    }
    if (i + TQ_RES_AHEAD < RF) load_res(i + TQ_RES_AHEAD, res8[i % TQ_RES_AHEAD]);
  }
}

// Panels of 16 columns of tiles, one after the other over all rows: 16 x 16 tiles of a panel at a time as eight
// 4 x 8 blocks, one per XCD, the panel's last rows and a narrower last panel row by row.  False: past the last tile.
__device__ __forceinline__ bool quad_panel(int p, int idx, int ncol, int nrow, int& bx, int& by) {
  const int w = min(TQ_PANEL, ncol - p * TQ_PANEL), i = idx & 255, round = idx >> 8;
  if (w < TQ_PANEL) {
    by = idx / w;
    bx = p * TQ_PANEL + idx - by * w;
    return by < nrow;
  }
  if ((round + 1) * 16 <= nrow) {
    const int xcd = i & 7, k = i >> 3;
    bx = p * TQ_PANEL + (xcd & 3) * 4 + (k & 3);
    by = round * 16 + (xcd >> 2) * 8 + (k >> 2);
  } else {
    bx = p * TQ_PANEL + (idx & (TQ_PANEL - 1));
    by = idx / TQ_PANEL;
  }
  return true;
}
// Tile t of a round of 256 regrouped (ncol, a and b are powers of two); the rows below the last whole round row by row.
__device__ __forceinline__ void quad_regroup(int t, int ncol, int nrow, int rm_a, int rm_r, int& bx, int& by) {
  const int cs = __builtin_ctz(ncol), as = __builtin_ctz(rm_a), round = t >> 8, i = t & 255;
  by = t >> cs;
  bx = t & (ncol - 1);
  if ((round + 1) * rm_r <= nrow) {  // a full round of 256 tiles
    const int xcd = i & 7, k = i >> 3, gs = cs - as;
    bx = ((xcd & ((1 << gs) - 1)) << as) + (k & (rm_a - 1));
    by = round * rm_r + (xcd >> gs) * (32 >> as) + (k >> as);
  }
}
// Tile t of ncol x nrow in the order of launch (see above: rm_a > 0 regrouped rounds, < 0 panels, 0 row by row).
__device__ __forceinline__ void quad_place(int t, int ncol, int nrow, int rm_a, int rm_r, int& bx, int& by) {
  if (rm_a < 0) {
    const int p = t / (TQ_PANEL * nrow);
    quad_panel(p, t - p * TQ_PANEL * nrow, ncol, nrow, bx, by);
  } else if (rm_a > 0) {
    quad_regroup(t, ncol, nrow, rm_a, rm_r, bx, by);
  } else {
    by = t / ncol;
    bx = t - by * ncol;
  }
}

// a group's last tile is as high as its rows need (48304 rows in 64 groups x 2816 x 4096 1154 -> 1125 us)
template <int MODE, int WF, bool ONCE>
__device__ __forceinline__ void quad_group_tile(const half_t* __restrict__ x, const void* __restrict__ Wp, int64_t M, int N, int K,
                                                int bx, int64_t m_own, const Epilogue& epi, const GroupTiles& gt) {
  if (M - m_own <= 128)
    quad_tile<MODE, WF, false, true, 4, false, ONCE>(x, Wp, M, N, K, bx, m_own, 0, epi, nullptr, 0, gt);
  else if (M - m_own <= 192)
    quad_tile<MODE, WF, false, true, 6, false, ONCE>(x, Wp, M, N, K, bx, m_own, 0, epi, nullptr, 0, gt);
  else
    quad_tile<MODE, WF, false, true, 8, false, ONCE>(x, Wp, M, N, K, bx, m_own, 0, epi, nullptr, 0, gt);
}

// ONCE of a grouped product: where an expert has one tile
template <int MODE, int WF, bool PART = false, bool GROUPED = false, int RF = 8, bool FEW = false, bool ONCE = false>
__global__ __launch_bounds__(TQ_THREADS) void linear_quad_kernel(
    const half_t* __restrict__ x, const void* __restrict__ Wp, int64_t M, int N, int K,
    int rm_a, int rm_r, Epilogue epi, float* __restrict__ part, int part_stages,
    GroupTiles gt = GroupTiles{}) {
  int bx = blockIdx.x, by = blockIdx.y;
  if constexpr (GROUPED) {
    const int ncol = gridDim.x, L = by * ncol + bx, total = *gt.n_tiles * ncol;
    const int per = (total + 7) / 8, t = (L & 7) * per + (L >> 3);
    if ((L >> 3) >= per || t >= total) return;
    by = t / ncol;
    bx = t - by * ncol;
    const int g = gt.tile_group[by];
    const int64_t first = gt.tile_row[by], end = gt.group_end[g], before = ONCE && g > 0 ? gt.group_end[g - 1] : 0;
    M = min(end, first + tq_bm(RF));
    Wp = (const char*)Wp + (int64_t)g * N * K * 2;
    if constexpr (ONCE)
      if (first == before && M == end) return quad_group_tile<MODE, WF, true>(x, Wp, M, N, K, bx, first, epi, gt);
    return quad_group_tile<MODE, WF, false>(x, Wp, M, N, K, bx, first, epi, gt);
  } else if (WF > 2 && rm_a < 0) {  // a row of the grid is a panel
    const int ncol = (N + tq_bn(WF) - 1) / tq_bn(WF), nrow = (int)((M + tq_bm(RF) - 1) / tq_bm(RF));
    if (!quad_panel(by, bx, ncol, nrow, bx, by)) return;
  } else if (rm_a > 0) {
    quad_regroup(by * gridDim.x + bx, gridDim.x, gridDim.y, rm_a, rm_r, bx, by);
  }
  if constexpr (!GROUPED)
    quad_tile<MODE, WF, PART, false, RF, FEW, ONCE>(x, Wp, M, N, K, bx, (int64_t)by * tq_bm(RF), blockIdx.z, epi, part, part_stages, gt);
}

// Tiles that would begin a round without filling half of it, in pieces: the first n_full tiles (of all K slices, whole
// rounds) are 256 x 256, the others PIECES = 2 of 256 x 128 or 4 of 128 x 128, side by side on one XCD.
template <int MODE, bool PART, int PIECES>
__global__ __launch_bounds__(TQ_THREADS) void linear_quad_pieces_kernel(
    const half_t* __restrict__ x, const void* __restrict__ Wp, int64_t M, int N, int K, int ncol, int nrow,
    int slices, int n_full, int rm_a, int rm_r, Epilogue epi, float* __restrict__ part, int part_stages) {
  const int tiles = ncol * nrow, j = (int)blockIdx.x - n_full;
  int unit = blockIdx.x, piece = 0, bx, by;
  if (j >= 0) {  // the first pieces of eight tiles, then their second ones, ...
    const int q = j / (8 * PIECES), w = min(8, tiles * slices - n_full - 8 * q), r = j % (8 * PIECES);
    unit = n_full + 8 * q + r % w;
    piece = r / w;
  }
  const int bz = PART ? unit / tiles : 0;
  quad_place(unit - bz * tiles, ncol, nrow, rm_a, rm_r, bx, by);
  const GroupTiles none{};
  const int64_t m_own = (int64_t)by * TQ_BM;
  if (j < 0) return quad_tile<MODE, 8, PART, false, 8, false>(x, Wp, M, N, K, bx, m_own, bz, epi, part, part_stages, none);
  bx = 2 * bx + (piece & 1);
  if (bx * tq_bn(4) >= N) return;
  if constexpr (PIECES == 2) {
    quad_tile<MODE, 4, PART, false, 8, false>(x, Wp, M, N, K, bx, m_own, bz, epi, part, part_stages, none);
  } else {
    const int64_t m = m_own + (piece >> 1) * tq_bm(4);
    if (m < M) quad_tile<MODE, 4, PART, false, 4, false>(x, Wp, M, N, K, bx, m, bz, epi, part, part_stages, none);
  }
}

// Rows cut evenly instead of by 256: the first n_tall rows of tiles are 32 RF high, the others 32 less (RF = 5 .. 8), at
// least 256 rows in all.
template <int MODE, int WF, bool PART, int RF>
__global__ __launch_bounds__(TQ_THREADS) void linear_quad_even_kernel(
    const half_t* __restrict__ x, const void* __restrict__ Wp, int64_t M, int N, int K, int nrow, int n_tall, int rm_a,
    int rm_r, Epilogue epi, float* __restrict__ part, int part_stages) {
  int bx = blockIdx.x, by = blockIdx.y;
  if (rm_a < 0) {
    if (!quad_panel(by, bx, (N + tq_bn(WF) - 1) / tq_bn(WF), nrow, bx, by)) return;
  } else if (rm_a > 0) {
    quad_regroup(by * gridDim.x + bx, gridDim.x, nrow, rm_a, rm_r, bx, by);
  }
  const GroupTiles none{};
  const int64_t m_own = (int64_t)(by * RF - max(by - n_tall, 0)) * 32;
  if (by < n_tall)
    quad_tile<MODE, WF, PART, false, RF, false>(x, Wp, M, N, K, bx, m_own, blockIdx.z, epi, part, part_stages, none);
  else
    quad_tile<MODE, WF, PART, false, RF - 1, false>(x, Wp, M, N, K, bx, m_own, blockIdx.z, epi, part, part_stages, none);
}

// ---- host side ------------------------------------------------------------------------------
// Per-device facts are kept per device: a process may drive several GPUs, from several threads.
constexpr int MAX_DEVICES = 64;
int current_device() {
  int dev = 0;
  return hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < MAX_DEVICES ? dev : -1;
}

std::atomic<int> g_num_cus[MAX_DEVICES];
int num_cus() {  // compute units of the current device
  const int dev = current_device();
  int n = dev >= 0 ? g_num_cus[dev].load(std::memory_order_relaxed) : 0;
  if (n == 0) {
    if (dev < 0 ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        n <= 0)
      n = 256;
    if (dev >= 0) g_num_cus[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Raises a kernel's dynamic LDS limit once per device (one mask per kernel instantiation; a
// second thread that gets here at the same time only repeats the call).  False: nothing may be launched; the
// runtime keeps the refusal as its last error, which every entry point reads behind its launches.
bool allow_lds(const void* kernel, int bytes, std::atomic<uint64_t>& done) {
  const int dev = current_device();
  const uint64_t bit = dev >= 0 ? 1ull << dev : 0;
  if (bit && (done.load(std::memory_order_acquire) & bit)) return true;
  if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess)
    return false;
  if (bit) done.fetch_or(bit, std::memory_order_release);
  return true;
}

template <int MB, bool W8, int MODE, bool XR = false>
void launch_stream_mb(const void* xp, const void* W, const void* scales, float* part, int S, int M,
                      int N, int K, int G, const Epilogue& epi, hipStream_t s, int64_t m_off = 0) {
  const int ntiles = N / 16, nks = K / 32;
  const int tiles_per_wg = (ntiles + G - 1) / G;
  const int gx = (ntiles + tiles_per_wg - 1) / tiles_per_wg;
  int ks_per_split = (nks + S - 1) / S;
  if (W8) ks_per_split = (ks_per_split + 1) & ~1;  // int8 blocks cover two steps
  // One or two tiles per workgroup (small models; split K): groups of as many.  A wider group's surplus slots
  // load the last tile again and multiply it: one row, 2304 x 768 4.6 -> 4.1 us, 2048 x 2048 in two
  // slices 4.7 -> 4.35, 6144 x 2048 7.2 -> 6.5, 768 x 3072 in two slices 5.9 -> 4.4.
  if constexpr (MB <= 2 && !XR && MODE != MODE_SELECT) {
    if (tiles_per_wg <= 2) {
      auto kernel = tiles_per_wg == 1 ? linear_stream_kernel<MB, W8, MODE, false, ST_KG, 1, 4>
                                      : linear_stream_kernel<MB, W8, MODE, false, ST_KG, 2, 4>;
      hipLaunchKernelGGL(kernel, dim3(gx, S), dim3(ST_KG * 64), 0, s, (const half_t*)xp, W, (const half_t*)scales,
                         part, M, N, K, tiles_per_wg, ks_per_split, epi, m_off);
      return;
    }
  }
  // Up to 32 packed rows: groups of 3 tiles instead of 4 when that needs no more groups (no
  // more sweeps over the activations) and leaves fewer empty tile slots, e.g. 3 tiles per
  // workgroup for qkv_proj at d_model 4096.
  if (MB <= 2 && !XR && (tiles_per_wg + 2) / 3 == (tiles_per_wg + 3) / 4 &&
      (tiles_per_wg + 2) / 3 * 3 < (tiles_per_wg + 3) / 4 * 4) {
    hipLaunchKernelGGL((linear_stream_kernel<(MB <= 2 ? MB : 1), W8, MODE, false, ST_KG, 3>),
                       dim3(gx, S), dim3(ST_KG * 64), 0, s, (const half_t*)xp, W,
                       (const half_t*)scales, part, M, N, K, tiles_per_wg, ks_per_split, epi,
                       m_off);
    return;
  }
  // The ragged bottom rows of a prefill-sized product (row-major activations, 33 .. 64 rows, fp16):
  // the workgroup's few tiles would leave most of the 8 tile slots per activation fragment empty
  // (their clamped loads still run), so groups of 4 are used when the tiles fit them.
  if constexpr (XR && !W8 && MB > 2) {
    if (tiles_per_wg <= ST_NT) {
      hipLaunchKernelGGL((linear_stream_kernel<MB, W8, MODE, XR, ST_KG, ST_NT>), dim3(gx, S),
                         dim3(ST_KG * 64), 0, s, (const half_t*)xp, W, (const half_t*)scales, part,
                         M, N, K, tiles_per_wg, ks_per_split, epi, m_off);
      return;
    }
  }
  hipLaunchKernelGGL((linear_stream_kernel<MB, W8, MODE, XR>), dim3(gx, S), dim3(ST_KG * 64), 0,
                     s, (const half_t*)xp, W, (const half_t*)scales, part, M, N, K, tiles_per_wg,
                     ks_per_split, epi, m_off);
}

constexpr int SH_GROUP = 12;  // most tiles per pass of the shared-activation kernel (4 lanes x 3)
// int8 only: 6 lanes x 3, from 14 tiles on (40 / 64 rows, us, against two passes of twelve or, of 14 tiles, the stream kernel: 57344 x 4096
// 51 / 59 and 60 / 67, 65536 x 8192 100 / 117 and 123 / 136, 73728 x 12288 146 / 167 and 191 / 219)
constexpr int SH_GROUP_W8 = 18;
// A vocabulary of 16-bit weights (13 or 14 tiles per workgroup) is one pass of a wave per tile over all of K: no
// sums between waves, the fewest registers and so the most loads in flight.  Measured, 50272 x 4096, us: 8 rows 69
// -> 64, 32 rows 75 -> 65 (6.3 TB/s; both on the stream kernel before), 40 rows 75 -> 66, 64 rows 95 -> 66, 100 rows
// 116 -> 93; K = 2048, 64 rows 48 -> 36; K = 9216, 64 rows 199 -> 138.  A third weight stage in flight costs as much as
// it gives (69 at 64 rows), eight K steps to a stage spill (89).  These are the numbers of tiles that gain at every number
// of rows.  A wave per tile for others, as they run now and so (K = 4096): 9 tiles, 1 row 44 and 46, 64 rows 53 and 50,
// 100 rows 67 and 71; 12 tiles 60 and 66, 70 and 69, 71 and 78; 15 tiles 73 and 76, 106 and 80, 129 and 99; 16 tiles 78
// and 90, 108 and 91, 127 and 102: less work in flight per CU below 13, and from 15 on four or more waves to a SIMD whose
// registers hold fewer loads each.
constexpr bool vocabulary_tiles(int tiles_per_wg) { return tiles_per_wg == 13 || tiles_per_wg == 14; }

// The shared-activation kernel sweeps K once per pass of SH_GROUP tiles: it is used when the
// workgroup's tiles fill their passes to at least three quarters.
bool share_fits(int tpw, bool w8) {
  if (tpw <= SH_GROUP) return true;  // one pass, with the tile count per wave chosen to fit
  if (w8 && tpw <= SH_GROUP_W8 && 4 * tpw >= 3 * SH_GROUP_W8) return true;  // one pass of 18
  const int passes = (tpw + SH_GROUP - 1) / SH_GROUP;
  return 4 * tpw >= 3 * passes * SH_GROUP;
}

template <int MB, bool W8, int MODE, int KL, int NG, int NT, int U, int PF = 2>
void launch_share_cfg(const void* xp, const void* W, const void* scales, float* part, int S, int M,
                      int N, int K, int tiles_per_wg, int gx, int ks_per_split, const Epilogue& epi,
                      hipStream_t s) {
  using C = ShareCfg<MB, W8, KL, NG, NT, U>;
  static std::atomic<uint64_t> lds_allowed{0};  // one mask per instantiation
  if (!allow_lds((const void*)linear_share_kernel<MB, W8, MODE, KL, NG, NT, U, PF>, C::LDS_BYTES,
                 lds_allowed))
    return;  // the caller's launch check reports the error
  hipLaunchKernelGGL((linear_share_kernel<MB, W8, MODE, KL, NG, NT, U, PF>), dim3(gx, S),
                     dim3(C::THREADS), C::LDS_BYTES, s, (const half_t*)xp, W,
                     (const half_t*)scales, part, M, N, K, tiles_per_wg, ks_per_split, epi);
}

// Tiles of a workgroup that the queue kernel takes: up to nine, as many as fit its sums beside their rows.  Up to 32 rows only from five
// tiles on, of int8 weights or two row blocks: the stream kernel loads four tiles' operands in one pass and does not go through
// LDS (us, stream and queue: 16384 x 4096, 32 rows 24.5 and 25, int8 17.3 and 18.2, 8 rows int8 16.9 and 18.1; five tiles int8
// 8 x 20480 x 5120 23.0 and 18.6; fp16 of one row block, seven tiles, 62.0 and 62.6).
constexpr int QUEUE_TILES = 9;
constexpr int queue_rows(int M) { return (M + 15) / 16; }  // row blocks that it multiplies, of eight from 65 rows on
constexpr bool queue_takes(int M, bool w8, int tiles_per_wg) {
  const int mb = queue_rows(M);
  if (tiles_per_wg > QUEUE_TILES || mb * tiles_per_wg > 64) return false;  // 64: QueueCfg::SUMS_FIT
  return mb > 2 || (tiles_per_wg >= 5 && (w8 || mb == 2));
}

}  // namespace
// (gemm_queue.h; compiled in files of its own, gemm_queue_*.hip)
template <bool W8, int MODE>
void launch_queue(const void* xp, const void* W, const void* scales, float* part, int S, int M, int N, int K,
                  int tiles_per_wg, const Epilogue& epi, hipStream_t s);
template <int MODE>
void launch_queue_rows(const void* x, const void* W, float* part, int S, int M, int N, int K, int tiles_per_wg,
                       const Epilogue& epi, hipStream_t s);
namespace {

// The shared-activation kernel: 33 .. 64 packed rows of more tiles than the queue kernel takes, and vocabularies from one row on,
// selections too (any number of tiles is right, in as many passes).
template <int MB, bool W8, int MODE>
void launch_share(const void* xp, const void* W, const void* scales, float* part, int S, int M,
                  int N, int K, int G, const Epilogue& epi, hipStream_t s) {
  const int ntiles = N / 16, nks = K / 32;
  const int tiles_per_wg = (ntiles + G - 1) / G;
  const int gx = (ntiles + tiles_per_wg - 1) / tiles_per_wg;
  int ks_per_split = (nks + S - 1) / S;
  if (W8) ks_per_split = (ks_per_split + 1) & ~1;  // int8 blocks cover two steps
  if constexpr (!W8) {
    if (MB <= 2 || MODE == MODE_SELECT || vocabulary_tiles(tiles_per_wg))
      return launch_share_cfg<MB, W8, MODE, 1, 14, 1, 4>(xp, W, scales, part, S, M, N, K, tiles_per_wg, gx, ks_per_split,
                                                         epi, s);
  }
  if constexpr (MB > 2 && MODE != MODE_SELECT) {
    if constexpr (W8) {
      if (tiles_per_wg > 12 && tiles_per_wg <= 18)
        return launch_share_cfg<MB, W8, MODE, 2, 6, 3, 2, 3>(xp, W, scales, part, S, M, N, K, tiles_per_wg, gx,
                                                             ks_per_split, epi, s);
    }
    launch_share_cfg<MB, W8, MODE, 2, 4, 3, 4>(xp, W, scales, part, S, M, N, K, tiles_per_wg, gx, ks_per_split, epi, s);
  } else {
    static_assert(!W8, "int8 weights of so few rows stream");
  }
}

// 65 .. 128 packed rows (eight row blocks) of more tiles than the queue kernel takes: the shared-activation kernel as 2 K
// lanes x 4 tile lanes with stages of two K steps; a vocabulary of 16-bit weights a wave per tile (50272 x 4096 at 128 rows
// 116 -> 95 us).
template <bool W8, int MODE>
void launch_wide(const void* xp, const void* W, const void* scales, float* part, int S, int M,
                 int N, int K, int G, const Epilogue& epi, hipStream_t s) {
  const int ntiles = N / 16, nks = K / 32;
  const int tiles_per_wg = (ntiles + G - 1) / G;
  const int gx = (ntiles + tiles_per_wg - 1) / tiles_per_wg;
  int ks_per_split = (nks + S - 1) / S;
  if (W8) ks_per_split = (ks_per_split + 1) & ~1;  // int8 blocks cover two steps
  if constexpr (!W8) {
    // (results of 16 bits only: its one chain over K has 1.4 times the error of two K lanes, K = 4096 3.9e-7 and 2.7e-7.
    // fp32 results of 128 rows by two K lanes: 50272 x 4096 114 us, by the chain 99.)
    if constexpr (!is_bf<MODE>) {
      if (vocabulary_tiles(tiles_per_wg) && !part)
        return tiles_per_wg == 13 ? launch_share_cfg<8, W8, MODE, 1, 13, 1, 2>(xp, W, scales, part, S, M, N, K,
                                                                               tiles_per_wg, gx, ks_per_split, epi, s)
                                  : launch_share_cfg<8, W8, MODE, 1, 14, 1, 2>(xp, W, scales, part, S, M, N, K,
                                                                               tiles_per_wg, gx, ks_per_split, epi, s);
    }
  }
  launch_share_cfg<8, W8, MODE, 2, 4, 3, 2, 2>(xp, W, scales, part, S, M, N, K, tiles_per_wg, gx, ks_per_split, epi, s);
}

// the tail in front of a product of at most LN_MAX_ROWS rows (S = 1, 2 or 4 slices); false: the LDS was refused
template <bool W8, int MODE, int S>
bool launch_stream_ln(const LnTail& ln, const void* W, const void* scales, int M, int N, int K, const Epilogue& epi,
                      hipStream_t s) {
  const int ntiles = N / 16, cus = num_cus(), tpw = (ntiles + cus - 1) / cus, gx = (ntiles + tpw - 1) / tpw;
  const int bytes = K * 32;
  static_assert(LN_MAX_K / 32 < 256 && LN_MAX_ROWS < 256, "packed below");
#define LN_RUN(NT)                                                                                            \
  do {                                                                                                        \
    auto kernel = linear_stream_ln_kernel<W8, MODE, NT, S>;                                                   \
    static std::atomic<uint64_t> allowed{0};                                                                  \
    if (!allow_lds((const void*)kernel, LN_MAX_K * 32, allowed)) return false;                                \
    hipLaunchKernelGGL(kernel, dim3(gx), dim3(ST_KG * 64), bytes, s, ln.part, ln.x, W, ln.bias, ln.gamma,     \
                       ln.beta, (uint32_t)ntiles << 8 | K / 32, (uint32_t)tpw << 8 | M, ln.x_out,             \
                       (const half_t*)scales, ln.eps, epi);                                                   \
  } while (0)
  if (tpw == 1) LN_RUN(1);
  else if (tpw == 2) LN_RUN(2);
  else if (tpw == 3 || tpw == 6) LN_RUN(3);
  else LN_RUN(4);
#undef LN_RUN
  return true;
}
template <bool W8, int MODE>
bool launch_stream_ln(const LnTail& ln, int S, const void* W, const void* scales, int M, int N, int K,
                      const Epilogue& epi, hipStream_t s) {
  return S == 1   ? launch_stream_ln<W8, MODE, 1>(ln, W, scales, M, N, K, epi, s)
         : S == 2 ? launch_stream_ln<W8, MODE, 2>(ln, W, scales, M, N, K, epi, s)
                  : launch_stream_ln<W8, MODE, 4>(ln, W, scales, M, N, K, epi, s);
}

template <bool W8, int MODE, bool XR = false>
void launch_stream(const void* xp, const void* W, const void* scales, float* part, int S, int M,
                   int N, int K, const Epilogue& epi, hipStream_t s, int64_t m_off = 0) {
  // (the runtime is asked for the device once: 125m, one row, 268 us a step, with two more questions to a product 278)
  const int cus = num_cus(), G = cus / S < 1 ? 1 : cus / S, tpw = (N / 16 + G - 1) / G;
  if constexpr (!XR && MODE != MODE_SELECT) {
    if (queue_takes(M, W8, tpw)) return launch_queue<W8, MODE>(xp, W, scales, part, S, M, N, K, tpw, epi, s);
    if (M > 64) return launch_wide<W8, MODE>(xp, W, scales, part, S, M, N, K, G, epi, s);
  }
  if constexpr (!XR && !W8) {
    if (M <= 64 && vocabulary_tiles(tpw)) {
      if (M > 48) return launch_share<4, W8, MODE>(xp, W, scales, part, S, M, N, K, G, epi, s);
      if (M > 32) return launch_share<3, W8, MODE>(xp, W, scales, part, S, M, N, K, G, epi, s);
      if (M > 16) return launch_share<2, W8, MODE>(xp, W, scales, part, S, M, N, K, G, epi, s);
      return launch_share<1, W8, MODE>(xp, W, scales, part, S, M, N, K, G, epi, s);
    }
  }
  if (!XR && MODE != MODE_SELECT && M > 32 && share_fits(tpw, W8)) {
    constexpr int PM = MODE == MODE_SELECT ? MODE_PLAIN : MODE;
    if (M > 48)
      launch_share<4, W8, PM>(xp, W, scales, part, S, M, N, K, G, epi, s);
    else
      launch_share<3, W8, PM>(xp, W, scales, part, S, M, N, K, G, epi, s);
    return;
  }
  switch ((M + 15) / 16) {
    case 1:
      launch_stream_mb<1, W8, MODE, XR>(xp, W, scales, part, S, M, N, K, G, epi, s, m_off);
      break;
    case 2:
      launch_stream_mb<2, W8, MODE, XR>(xp, W, scales, part, S, M, N, K, G, epi, s, m_off);
      break;
    case 3:
      launch_stream_mb<3, W8, MODE, XR>(xp, W, scales, part, S, M, N, K, G, epi, s, m_off);
      break;
    default:
      launch_stream_mb<4, W8, MODE, XR>(xp, W, scales, part, S, M, N, K, G, epi, s, m_off);
      break;
  }
}

// Row by row, a round of 256 tiles over more than 64 columns leaves each XCD a strip of at least eight columns
// and a row or two, whose weights come from beyond its L2 (197 columns, the vocabulary: 25 strips of
// weights and 2 of activations per XCD and round, 4.3 TB/s; in panels 4 and 8).  Measured, 32800 x
// 50272 x 4096 12.3 -> 10.7 ms, 6038 rows with fp32 results 2372 -> 1963 us, 2005 rows 807 -> 685, 1500
// rows 600 -> 502; 6038 x 21888 x 4096 (86 columns) 960 -> 918; 48 and 64 columns are the same either way.
bool wide_panels(int ncol) { return ncol > 64; }

// regrouping of a round's 256 tiles: a x b per XCD with a * b = 32, (ncol / a) * (r / b) = 8 for r = 256 / ncol
// rows per round; taken when it beats the default strip (ncol / 8) x r.  a < 0: panels, a = 0: row by row, which is
// also the order of a single row and of less than one round
struct TileOrder {
  int a, r;
};
// (256 x 64 tiles, rarely more than a round, are not taken in panels: code in front of the first load shows in
// products of 5 us)
TileOrder tile_order(int ncol, int nrow, int WF) {
  TileOrder o{0, 0};
  if (nrow == 1) return o;
  if (WF > 2 && wide_panels(ncol)) {
    o.a = -TQ_PANEL;
  } else if (ncol >= 8 && 256 % ncol == 0 && 256 / ncol <= nrow) {
    const int r = 256 / ncol;
    int best = ncol / 8 + r;
    for (int a = 1; a <= 32; a *= 2) {
      const int b = 32 / a;
      if (ncol % a || r % b || (ncol / a) * (r / b) != 8) continue;
      if (a + b < best) best = a + b, o = TileOrder{a, r};
    }
  }
  return o;
}
dim3 quad_grid(int ncol, int nrow, const TileOrder& o, int slices = 1) {
  return o.a < 0 ? dim3(TQ_PANEL * nrow, (ncol + TQ_PANEL - 1) / TQ_PANEL, slices) : dim3(ncol, nrow, slices);
}

// Time of a tile of 32 RF rows and 32 WF columns while the whole chip computes such tiles, us; of a round that
// fills a part of it: the clock rises as CUs fall idle (K = 16384, 256 x 256 tiles on 256, 192 and 128 CUs 382, 325 and
// 277 us).  Fitted to 1200 products of 260 .. 6038 rows (K = 768 .. 16384), which it meets within 5 % (rms).
double quad_tile_us(int WF, int RF, int K) {
  if (WF == 2) return 4.3 + 0.0088 * K;
  return WF == 8 ? 1.0 + 1.45 * RF + (0.0063 + 0.00165 * RF) * K : 0.8 + 0.75 * RF + (0.0024 + 0.00127 * RF) * K;
}
double quad_part_round(int tiles, int cus) { return 0.75 + 0.25 * tiles / cus; }
double quad_rounds_us(int64_t tiles, double tile_us, int cus) {
  const int left = (int)(tiles % cus);
  return tile_us * ((double)(tiles / cus) + (left ? quad_part_round(left, cus) : 0.0));
}
// Into how many pieces the tiles are cut that are left after whole rounds of 256 x 256 ones (1: they are not): as many
// as still run in one round.  Without and with, K = 4096, us: 2005 x 9216 (32 tiles left) 170 -> 130 in quarters,
// 147 in halves; 2005 x 10240 (64) 171 -> 136, 149; 1500 x 14848 (92) 198 -> 171; 2005 x 12288 (128) 179 ->
// 162, 171 in quarters; 6038 x 5888 (two rounds and 40) 272 -> 233; 2005 x 50272 (six and 40) 677 -> 638.
// More than half a round is not cut: 1500 x 50272 (four and 158) 490 and 502.
int quad_pieces(int64_t tiles, int cus) {
  const int64_t left = tiles % cus;
  return tiles < cus || left == 0 || left * 2 > cus ? 1 : left * 4 > cus ? 2 : 4;
}
double quad_cost(int64_t tiles, int K, int cus) {  // 256 x 256 tiles, us
  const int pieces = quad_pieces(tiles, cus);
  if (pieces == 1) return quad_rounds_us(tiles, quad_tile_us(8, 8, K), cus);
  return (double)(tiles / cus) * quad_tile_us(8, 8, K) +
         quad_rounds_us(tiles % cus * pieces, quad_tile_us(4, pieces == 2 ? 8 : 4, K), cus);
}

// The cheapest even cut of at least 256 rows (linear_quad_even_kernel): as many rows of tiles as fill whole rounds,
// each of the height that is left for it, so that neither a round is left half empty nor a row of tiles.  Up to 24 rounds
// (100 of them are 0.01 % better) and 16384 rows (beyond, 0.7 % on average, for a choice of 3 us and more on the host;
// 0.06 us at 300 rows, 0.2 at 2000, 0.5 at 5000).  Of 19200 products of eight widths from 768 to 9216 and 256 to 16384
// rows 56 % are cut evenly; by columns x rows of the taller tiles, how often and what the price loses without them, on average and at most: 128
// x 160 13 % (2.2, 53), x 192 3 (0.4, 24), x 224 3 (0.2, 12), 256 x 160 8 (0.8, 20), x 192 7 (0.6, 22), x 224 10 (0.6, 15), x 256 11 (0.2, 7).
// Against tiles of one height (256 rows, or 128 x 128), us: 300 x 16384 x 4096 68 -> 50, 640 x 12288 x 4096 80 -> 67, 900 x
// 16384 x 4096 110 -> 97, 1100 x 4096 x 4096 53 -> 40, 1260 x 4096 x 16384 201 -> 167, 1607 x 16384 x 4096 in a model 211 ->
// 180, 2140 x 2048 x 8192 101 -> 75, 2460 x 4096 x 16384 328 -> 252, 1390 x 6144 x 2048 61 -> 37; 360 products of 66 ..
// 8300 rows (K = 768 .. 16384) 4 % on average, none slower than the runs of one side differ.
struct QuadPlan {
  double us = 1e30;
  int wf = 0, rf = 0, nrow = 0, n_tall = 0;
};
QuadPlan quad_plan(int64_t M, int N, int K, int S, int cus) {
  QuadPlan best;
  if (M < TQ_BM || M > 16384) return best;
  const int units = (int)((M + 31) / 32), most = 24 * cus;
  for (int wf = 4; wf <= 8; wf += 4) {
    const int ncol = (N + tq_bn(wf) - 1) / tq_bn(wf);
    // (128 columns: 256-row tiles among lower ones are never the cheapest)
    for (int nrow = (units + wf / 4 + 5) / (wf / 4 + 6); nrow * 4 < units + 4; ++nrow) {
      const int rf = nrow * 4 < units ? (units + nrow - 1) / nrow : 5;  // (the last: all rows 128 high)
      const int n_tall = nrow * 4 < units ? units - nrow * (rf - 1) : 0;
      if ((int64_t)nrow * ncol * S > most) break;
      const int slice = nrow * ncol, tiles = slice * S;
      const double tall = quad_tile_us(wf, rf, K / S), low = quad_tile_us(wf, rf - 1, K / S);
      double us = 0;
      for (int t = 0; t < tiles && us < best.us; t += cus) {  // a round takes as long as its tallest tile
        const int n = tiles - t < cus ? tiles - t : cus, at = S == 1 ? t : t % slice;
        us += (at < n_tall * ncol || (n_tall && at + n > slice) ? tall : low) * (n < cus ? quad_part_round(n, cus) : 1.0);
      }
      if (us < best.us) best = QuadPlan{us, wf, rf, nrow, n_tall};
    }
  }
  return best;
}
// The cheapest form of S sums over at least 256 rows: 256 x 256 tiles, the last of them in pieces (w = 8), 256 x
// 128 (4), 256 x 64 (2), or an even cut.
constexpr int QUAD_EVEN = 1;
struct QuadPrice {
  double us;
  int w;
  QuadPlan even;
};
QuadPrice quad_price(int64_t M, int N, int K, int S, int cus) {
  const int64_t rows = (M + TQ_BM - 1) / TQ_BM * S;
  QuadPrice best{quad_cost(rows * ((N + 255) / 256), K / S, cus), 8, quad_plan(M, N, K, S, cus)};
  const double four = quad_rounds_us(rows * ((N + 127) / 128), quad_tile_us(4, 8, K / S), cus);
  const double two = quad_rounds_us(rows * ((N + 63) / 64), quad_tile_us(2, 8, K / S), cus);
  if (four < best.us) best.us = four, best.w = 4;
  if (two < best.us) best.us = two, best.w = 2;
  if (best.even.us < best.us) best.us = best.even.us, best.w = QUAD_EVEN;
  return best;
}
// Row by row, a number of columns that 4 does not divide moves a column on to another XCD in each row of tiles, and each of
// them reads its weights from beyond its own L2; an even cut has many rows.  In panels a column keeps to one XCD: 516 x
// 11392 x 1984 (45 columns, five rows) 40.3 -> 35.5 us, 1143 x 2160 x 1856 (17, nine) 19.2 -> 16.9, 669 x 12480 x 512 21.1 ->
// 16.2.  28 columns, two XCDs to each, are as well row by row (1436 x 3552 x 448 10.0 and 10.7).  The empty places behind the
// tiles of a slice leave the XCDs unequal shares: slices are taken so where all tiles still run at once (in two slices, 600 x
// 3424 x 9600 55.4 -> 51.1; 778 x 1600 x 14720 64 and 76).
TileOrder even_order(int ncol, int nrow, int WF, int S, int cus) {
  TileOrder o = tile_order(ncol, nrow, WF);
  if (o.a == 0 && ncol % 4 && ncol > TQ_PANEL && nrow > 1 && (S == 1 || (ncol * nrow + 7) / 8 * 8 * S <= cus)) o.a = -TQ_PANEL;
  return o;
}
template <int MODE, int WF, bool PART, int RF>
void launch_quad_even(const void* x, const void* W, int64_t M, int N, int K, int S, const QuadPlan& p,
                      const Epilogue& epi, float* part, hipStream_t s) {
  static std::atomic<uint64_t> lds_allowed_e{0};
  constexpr int lds = tq_lds_bytes(WF, RF) > tq_lds_bytes(WF, RF - 1) ? tq_lds_bytes(WF, RF) : tq_lds_bytes(WF, RF - 1);
  auto kernel = linear_quad_even_kernel<MODE, WF, PART, RF>;
  if (!allow_lds((const void*)kernel, lds, lds_allowed_e)) return;
  const int ncol = (N + tq_bn(WF) - 1) / tq_bn(WF);
  const TileOrder o = even_order(ncol, p.nrow, WF, S, num_cus());
  hipLaunchKernelGGL(kernel, quad_grid(ncol, p.nrow, o, S), dim3(TQ_THREADS), lds, s, (const half_t*)x, W, M, N, K,
                     p.nrow, p.n_tall, o.a, o.r, epi, part, K / 64 / S);
}
template <int MODE, bool PART>
void launch_quad_plan(const void* x, const void* W, int64_t M, int N, int K, int S, const QuadPlan& p,
                      const Epilogue& epi, float* part, hipStream_t s) {
  if (p.wf == 8) {
    if (p.rf == 8) return launch_quad_even<MODE, 8, PART, 8>(x, W, M, N, K, S, p, epi, part, s);
    if (p.rf == 7) return launch_quad_even<MODE, 8, PART, 7>(x, W, M, N, K, S, p, epi, part, s);
    if (p.rf == 6) return launch_quad_even<MODE, 8, PART, 6>(x, W, M, N, K, S, p, epi, part, s);
    return launch_quad_even<MODE, 8, PART, 5>(x, W, M, N, K, S, p, epi, part, s);
  }
  if (p.rf == 7) return launch_quad_even<MODE, 4, PART, 7>(x, W, M, N, K, S, p, epi, part, s);
  if (p.rf == 6) return launch_quad_even<MODE, 4, PART, 6>(x, W, M, N, K, S, p, epi, part, s);
  return launch_quad_even<MODE, 4, PART, 5>(x, W, M, N, K, S, p, epi, part, s);
}

template <int MODE, bool PART, int PIECES>
void launch_quad_pieces(const void* x, const void* W, int64_t M, int N, int K, int S, const Epilogue& epi, float* part,
                        hipStream_t s) {
  static std::atomic<uint64_t> lds_allowed_h{0};
  auto kernel = linear_quad_pieces_kernel<MODE, PART, PIECES>;
  if (!allow_lds((const void*)kernel, tq_lds_bytes(8), lds_allowed_h)) return;
  const int ncol = (N + tq_bn(8) - 1) / tq_bn(8), nrow = (int)((M + TQ_BM - 1) / TQ_BM), units = ncol * nrow * S;
  const int n_full = units / num_cus() * num_cus();
  const TileOrder o = tile_order(ncol, nrow, 8);
  hipLaunchKernelGGL(kernel, dim3(n_full + PIECES * (units - n_full)), dim3(TQ_THREADS), tq_lds_bytes(8), s,
                     (const half_t*)x, W, M, N, K, ncol, nrow, S, n_full, o.a, o.r, epi, part, K / 64 / S);
}

// One launch of the four-wave kernel (WF = 8: 256 x 256 tiles, the last of them in pieces where that pays; WF = 4:
// 256 x 128, WF = 2: 256 x 64) on rows 0 .. M_main - 1 (a ragged last row tile is moved up) plus the streaming kernel on the rows from
// M_main on (at most 128).
template <int MODE, int WF>
void launch_quad(const void* x, const void* W, const void* scales, int64_t M, int64_t M_main, int N,
                 int K, int pieces, const Epilogue& epi, hipStream_t s) {
  const int ncol = (N + tq_bn(WF) - 1) / tq_bn(WF);
  const int nrow = (int)((M_main + TQ_BM - 1) / TQ_BM);
  if (pieces == 4) {
    launch_quad_pieces<MODE, false, 4>(x, W, M_main, N, K, 1, epi, nullptr, s);
  } else if (pieces == 2) {
    launch_quad_pieces<MODE, false, 2>(x, W, M_main, N, K, 1, epi, nullptr, s);
  } else {
    static std::atomic<uint64_t> lds_allowed_q[2] = {};
    auto kernel = nrow == 1 ? linear_quad_kernel<MODE, WF, false, false, 8, false, true>
                            : linear_quad_kernel<MODE, WF, false, false, 8, false, false>;
    if (!allow_lds((const void*)kernel, tq_lds_bytes(WF), lds_allowed_q[nrow == 1])) return;
    const TileOrder o = tile_order(ncol, nrow, WF);
    hipLaunchKernelGGL(kernel, quad_grid(ncol, nrow, o), dim3(TQ_THREADS),
                       tq_lds_bytes(WF), s, (const half_t*)x, W, M_main, N, K, o.a, o.r, epi,
                       (float*)nullptr, 0, GroupTiles{});
  }
  for (int64_t m0 = M_main; m0 < M; m0 += 64)
    launch_stream<false, MODE, true>(x, W, scales, nullptr, 1, (int)min((int64_t)64, M - m0), N,
                                     K, epi, s, m0);
}

// One round of tiles over fewer rows than a 256-row tile holds, or a little more than one of 128.
//   RF = 4: 128 x 128 tiles, two rows of them side by side on one XCD (also of more rows, where one round of them
//   is cheapest: 2048 x 2048 x 4096 44.9 us on 256 x 64 tiles -> 39.6).  Of 129 .. 256 rows a CU then reads half as
//   many activations as with the 256 x 64 form, its weights once more from L2: 200 x 12288 x 4096 43.3 ->
//   37.5 us, 200 x 16384 x 4096 48.1 -> 41.2, 130 x 8192 x 2048 21.8 -> 18.7.  (As split-K sums they
//   gained nothing: 200 x 4096 x 16384 49.8 -> 53.5.)  Of 129 .. 256 rows its longer fill of the rings is paid back from
//   K = 512 on (200 x 4096: K = 256 7.0 -> 7.1 us, 512 9.0 -> 8.6), with more than 192 tiles from K = 4096 on (160 x
//   16384: K = 2048 26.1 -> 27.1, 4096 47 -> 42).
//   WF = 8: 128 to 256 rows x 256 tiles that repeat the last row, for outputs wide enough that one row of them fills
//   the chip (the vocabulary): bf16 200 x 50272 x 4096 168 -> 101 us.  As high as the rows need, fp16, against 256 rows: 66
//   106 -> 86, 129 106 -> 89, 170 111 -> 95, 200 111 -> 101.
template <int MODE, int WF, int RF>
void launch_few_rows(const void* x, const void* W, int64_t M, int N, int K, const Epilogue& epi, hipStream_t s) {
  static std::atomic<uint64_t> lds_allowed_s{0};
  const int ncol = (N + tq_bn(WF) - 1) / tq_bn(WF), nrow = (int)((M + tq_bm(RF) - 1) / tq_bm(RF));
  constexpr bool ONCE = WF == 8;  // tiles of 256 columns are one row, the others two
  auto kernel = linear_quad_kernel<MODE, WF, false, false, RF, true, ONCE>;
  if (!allow_lds((const void*)kernel, tq_lds_bytes(WF, RF), lds_allowed_s)) return;
  const TileOrder o{nrow == 1 ? 0 : -TQ_PANEL, 0};
  hipLaunchKernelGGL(kernel, quad_grid(ncol, nrow, o), dim3(TQ_THREADS), tq_lds_bytes(WF, RF), s, (const half_t*)x, W,
                     M, N, K, o.a, o.r, epi, (float*)nullptr, 0, GroupTiles{});
}

// Split-K launch of a four-wave form (WF = 2: 256 x 64 tiles, WF = 4: 256 x 128, WF = 8: 256 x 256, of at least
// 256 rows) on row-major activations: S slices of K, each a whole number of 64-wide stages (at least two),
// fp32 sums into part[S][M][N].
template <int MODE, int WF>
void launch_quad_partial_w(const void* x, const void* W, float* part, int64_t M, int N, int K,
                           int S, hipStream_t s) {
  static std::atomic<uint64_t> lds_allowed_p{0};
  auto kernel = linear_quad_kernel<MODE, WF, true>;
  if (!allow_lds((const void*)kernel, tq_lds_bytes(WF), lds_allowed_p)) return;
  const int ncol = (N + tq_bn(WF) - 1) / tq_bn(WF);
  const int nrow = (int)((M + TQ_BM - 1) / TQ_BM);
  Epilogue e{};
  const TileOrder o = tile_order(ncol, nrow, WF);
  hipLaunchKernelGGL(kernel, quad_grid(ncol, nrow, o, S), dim3(TQ_THREADS), tq_lds_bytes(WF), s,
                     (const half_t*)x, W, M, N, K, o.a, o.r, e, part, K / 64 / S, GroupTiles{});
}

// How a product of more than 64 row-major rows is taken: the forms of quad_price, 128 x 128 tiles (w = 0), and two ways
// to take a ragged bottom of at most 128 rows: as one more, moved-up row of tiles, or (main < M) through the
// streaming kernel, a sweep over the weights per 64 rows.
struct TileChoice {
  double us;
  int w;
  int64_t main;
  QuadPlan even;
};
TileChoice tile_choice(int64_t M, int N, int K, int cus) {
  const int64_t rows = (M + TQ_BM - 1) / TQ_BM, rem = M % TQ_BM;
  const int64_t cols[3] = {(N + 255) / 256, (N + 127) / 128, (N + 63) / 64};
  TileChoice best{quad_rounds_us(rows * cols[2], quad_tile_us(2, 8, K), cus), 2, M, QuadPlan{}};
  auto offer = [&](double us, int w, int64_t m_main) {
    if (us < best.us) best.us = us, best.w = w, best.main = m_main;
  };
  if (M > TQ_BM) {
    const int64_t tiles = (M + 127) / 128 * cols[1];
    // An odd number of 128 rows, the last of them nearly full (a 256-row tile would repeat its last row
    // there, from the CU's own cache): 384 x 4096 x 16384 (96 tiles) 139 us against 133 on 256 x 64, 640
    // 140 against 136, but 384 x 7168 x 28672 (168) 248 against 297; of more than a round bf16 352 x
    // 50272 x 768 55 against 51 on 256 x 256, 384 x 50272 x 4096 197 against 186, 300 rows 173 against 184.
    const bool full = rem >= 96 && rem <= 128;
    const double more = !full ? 1.0 : K > 8192 && tiles * 8 <= cus * 5 ? 1.25 : 1.12;
    offer(quad_rounds_us(tiles, quad_tile_us(4, 4, K), cus) * more, 0, M);
  }
  if (M >= TQ_BM) {
    const QuadPrice p = quad_price(M, N, K, 1, cus);
    best.even = p.even;
    offer(p.us, p.w, M);
  }
  if (rem > 0 && rem <= 128 && M - rem >= TQ_BM) {
    const double below = (double)((rem + 63) / 64) * ((double)N * K * 2 / 5e6 + 4);  // us of the streaming launches
    offer(quad_rounds_us((rows - 1) * cols[1], quad_tile_us(4, 8, K), cus) + below, 4, M - rem);
    offer(quad_cost((rows - 1) * cols[0], K, cus) + below, 8, M - rem);
  }
  return best;
}

// What a product of row-major activations is taken with.
struct TileForm {
  int kind = MSA_TILES_SIMPLE, wf = 4, rf = 4, pieces = 1;
  int64_t main = 0;  // rows in tiles; the others in sweeps over the weights
  int queue = 0;     // tiles of 16 columns to a workgroup of the queue kernel
  QuadPlan even;
};
// 129 .. 256 row-major rows in queues (gemm_queue.h): the tiles of a workgroup, 0 where there are more than five, or where
// K is not in whole slots.  Two workgroups share a column of them.
constexpr int QUEUE_ROWS_TILES = 5;
constexpr int queue_rows_blocks(int M) { return M <= 160 ? 5 : M <= 192 ? 6 : M <= 224 ? 7 : 8; }
int queue_rows_tiles(int64_t M, int N, int K, int S, int cus) {
  if (M <= 128 || M > 256 || K % 64 || K < 128) return 0;
  const int G = cus / (2 * S) < 1 ? 1 : cus / (2 * S), tiles = (N / 16 + G - 1) / G;
  return tiles <= QUEUE_ROWS_TILES ? tiles : 0;
}
// S sums to be stored as they are, of any number of rows: the cheapest form of quad_price.  Below 256 rows 256 x 64 tiles while
// their slices fit the chip in one round; an S beyond that means 256 x 128 tiles (pick_row_splits).
// Of 129 .. 256 rows queues where those tiles would leave more than a quarter of the chip idle (us, 200 rows: 2560 x 2560 in four
// slices, 160 tiles, 12.2 and 11.4 in queues, x 10240 30.2 and 23.3, 2048 x 2048 in four, 128 tiles, 10.1 and 8.9; 256 tiles:
// 2048 x 8192 in eight 17.2, in four in queues 18.0, 4096 x 4096 in four 17.2, in two in queues 17.9).
TileForm partial_form(int64_t M, int N, int K, int S, int cus) {
  const int64_t rows = (M + TQ_BM - 1) / TQ_BM;
  TileForm f;
  f.main = M, f.rf = 8;
  f.queue = rows * ((N + 63) / 64) * S * 4 <= cus * 3 ? queue_rows_tiles(M, N, K, S, cus) : 0;
  if (f.queue) {
    f.kind = MSA_TILES_QUEUE;
    return f;
  }
  if (M < TQ_BM) {
    f.kind = MSA_TILES_FEW;
    f.wf = rows * ((N + 63) / 64) * S > cus ? 4 : 2;
    return f;
  }
  const QuadPrice price = quad_price(M, N, K, S, cus);
  f.kind = price.w == QUAD_EVEN ? MSA_TILES_EVEN : MSA_TILES_WHOLE;
  f.even = price.even;
  f.wf = price.w == QUAD_EVEN ? price.even.wf : price.w;
  if (price.w == QUAD_EVEN) f.rf = price.even.rf;
  if (price.w == 8) f.pieces = quad_pieces(rows * ((N + 255) / 256) * S, cus);
  return f;
}
// A whole product.  Fewer rows than a tile, or hardly more: launch_few_rows where its tiles fill one round (three quarters of
// the CUs with 256 x 256 tiles).  Else the cheapest form of tile_choice; the 256 x 64 tiles also serve 65 .. 255
// rows (they repeat the last row instead of moving up).  linear_tiled_kernel is left with what is no
// multiple of 64 deep: a few tiles of the direct-to-LDS forms are ahead of it too (us: 100 x 768 x 768 17.0 and 10.1, 200
// x 1024 x 4096 60 and 28, 300 x 768 x 3072 58 and 22, 500 x 256 x 1024 20.5 and 11.2, 65 x 16 x 2048 29.8 and 18.5, 65
// x 128 x 128 8.0 and 7.6).
TileForm tile_form(int64_t M, int N, int K, int cus) {
  TileForm f;
  if (M <= 64) {
    f.kind = MSA_TILES_NONE;
    return f;
  }
  f.main = M;
  if (K % 64 || K < 128) return f;
  f.queue = queue_rows_tiles(M, N, K, 1, cus);
  if (f.queue) {
    f.kind = MSA_TILES_QUEUE;
    return f;
  }
  const int64_t cols[2] = {(N + 255) / 256, (N + 127) / 128};
  if (M < TQ_BM && cols[0] <= cus && cols[0] * 4 >= cus * 3) {
    f.kind = MSA_TILES_FEW;
    f.wf = 8, f.rf = M <= 128 ? 4 : M <= 160 ? 5 : M <= 192 ? 6 : M <= 224 ? 7 : 8;
    return f;
  }
  if (M > 128 && M <= TQ_BM && cols[1] * 2 <= cus && K >= (cols[1] * 8 <= cus * 3 ? 512 : 4096)) {
    f.kind = MSA_TILES_FEW;
    return f;
  }
  const TileChoice c = tile_choice(M, N, K, cus);
  f.kind = c.w == QUAD_EVEN ? MSA_TILES_EVEN : c.w == 0 ? MSA_TILES_FEW : MSA_TILES_WHOLE;
  f.even = c.even;
  f.main = c.w == QUAD_EVEN || c.w == 0 ? M : c.main;
  if (c.w == QUAD_EVEN) f.wf = c.even.wf, f.rf = c.even.rf;
  if (c.w > 1) f.wf = c.w, f.rf = 8;
  if (c.w == 8) f.pieces = quad_pieces((f.main + TQ_BM - 1) / TQ_BM * cols[0], cus);
  return f;
}

template <int MODE>
void launch_quad_partial(const void* x, const void* W, float* part, int64_t M, int N, int K, int S,
                         hipStream_t s) {
  const TileForm f = partial_form(M, N, K, S, num_cus());
  if (f.kind == MSA_TILES_QUEUE) return launch_queue_rows<MODE>(x, W, part, S, (int)M, N, K, f.queue, Epilogue{}, s);
  if (f.kind == MSA_TILES_EVEN) return launch_quad_plan<MODE, true>(x, W, M, N, K, S, f.even, Epilogue{}, part, s);
  if (f.pieces == 4) return launch_quad_pieces<MODE, true, 4>(x, W, M, N, K, S, Epilogue{}, part, s);
  if (f.pieces == 2) return launch_quad_pieces<MODE, true, 2>(x, W, M, N, K, S, Epilogue{}, part, s);
  if (f.wf == 8) return launch_quad_partial_w<MODE, 8>(x, W, part, M, N, K, S, s);
  if (f.wf == 4) return launch_quad_partial_w<MODE, 4>(x, W, part, M, N, K, S, s);
  launch_quad_partial_w<MODE, 2>(x, W, part, M, N, K, S, s);
}

// Slices for a product of M row-major rows whose tiles alone leave most of the chip idle (a
// decode batch of a few hundred rows against d_model output features): the most of 2, 4, 8 that
// keep the 256 x 64 tiles within the chip, the K range of a slice at 512 or more, and whole
// stages.  Where a slice would still span 4096 or more of K, twice the slices over 256 x 128
// tiles measured faster (half the activation bytes per workgroup and weight byte: M = 256,
// N = 4096, K = 16384: 51.8 against 55.4 us; M = 512: 78.0 against 93.6; M = 200, inside a
// decode step: 42.4 against 47.2).
int pick_row_splits(int64_t M, int N, int K) {
  if (M < 1 || N % 16 || K % 64) return 1;
  const int64_t tiles = ((M + TQ_BM - 1) / TQ_BM) * ((N + tq_bn(2) - 1) / tq_bn(2));
  const int cus = num_cus();
  int best = 1;
  for (int S = 2; S <= 8; S *= 2)
    if (tiles * S <= cus && K % (64 * S) == 0 && K / S >= 512) best = S;
  // in queues, half as many are as fast from 2048 columns or 4096 of K on, and leave the tail half as much to add (us, 200 rows: 2048 x
  // 2048 in four 8.9, in two 8.4, 2560 x 2560 11.4 and 11.1, 1024 x 4096 in eight 9.4, in four 8.4)
  if (best >= 4 && K / best <= 1024 && partial_form(M, N, K, best, cus).queue > 3 && partial_form(M, N, K, best / 2, cus).queue)
    return best / 2;
  if (best > 1 && best < 8 && M > 128 && K / best >= 4096 && K % (128 * best) == 0) best *= 2;
  return best;
}

// The same for fp16 prompts whose tail adds the slices: two of a long sum (K of 8192 or more) whose 256 x 256 tiles
// fill half of the chip or less.  One slice takes 256 x 128 tiles there, at 0.61 of the wide tiles' time for half of
// their work.  Product, tail and LayerNorm, cold weights, one slice and two, us: 4096 x 16384 over 1180 rows 205 and 166,
// 1692 225 and 200, 2048 250 and 224; 5120 x 20480 over 1024 257 and 215, 1536 289 and 263; 7168 x 28672 over 768 380 and
// 305, 1024 396 and 344; 9216 x 36864 over 512 481 and 370, 768 503 and 433; 9216 x 9216 over 512 128 and 108; 2560 x
// 10240 over 1692 135 and 113, 2304 141 and 123.  A sum shorter than 16384 stops at three quarters of that half: 2048
// x 8192 over 3072 rows (96 tiles) 120 and 109, 3328 122 and 116, 3584 125 and 122, 3840 128 and 129, 4096 135 and 133.
// (The line is drawn for K = 8192; between it and 16384 two slices stay ahead past it: 9216 x 9216 over 768 rows, 108
// tiles, 137 and 126, 2560 x 10240 over 3072, 120 tiles, 156 and 148.)  Where one slice would fit as 256 x 128 or 128 x 128
// tiles, two are taken if their price with what the second slice costs to write and read is the lower: 4096 x 16384, product
// alone, 520 rows 104 and 79, 700 118 and 90, 1000 144 and 117; 2048 x 8192 over 1100 rows 59 and 44, 1500 67 and 48.
int pick_row_splits_f16(int64_t M, int N, int K) {
  const int few = pick_row_splits(M, N, K);
  if (few > 1 || M < TQ_BM || N % 16 || K % 128 || K < 8192) return few;
  const int64_t rows = (M + TQ_BM - 1) / TQ_BM, tiles8 = rows * ((N + 255) / 256), tiles4 = rows * ((N + 127) / 128);
  if (tiles8 * 2 > num_cus() * (K >= 16384 ? 4 : 3) / 4) return 1;
  if (tiles4 * 2 > num_cus()) return 2;
  const double one = tile_choice(M, N, K, num_cus()).us, two = quad_price(M, N, K, 2, num_cus()).us;
  return two + (double)M * N * 8 / 5e6 < 0.95 * one ? 2 : 1;
}

// The same for sums that leave as fp32 from any width of tile (bf16): also two slices of prompts' products whose
// 256 x 256 tiles fill half of the chip or less, priced with what the second slice costs to write and read (5
// TB/s).  1500 x 4096 x 16384: one slice of 256 x 128 tiles 194 us, two of 256 x 256 165 and 5 in the tail; 1500 x
// 4096 x 4096 stays at one, 54 against 53 and 5, and so do 1000 x 4096 x 1024 (15.0 against 16.8 and 3) and 3000 x 1024
// x 1024 (14.3, 17.3 and 2.5), whose one slice is taken in 256 x 64 tiles; 1000 x 4096 x 4096 43 against 37 and 3.
// Where those tiles leave more than a quarter of the chip idle the clock is higher than the price's: up to K = 8192
// one slice (2048 x 1408 x 4096 36 against 40 and 2; 1000 x 2560 x 10240 99 against 68 and 2).
// (Rounds of whole tiles and of their pieces, at the costs below; the launch of either number of slices then takes the
// cheapest form of quad_price, even cuts among them: 520 to 800 x 4096 x 4096 stay at one slice, 31 us, where two would take 28.)
int pick_row_splits_f32(int64_t M, int N, int K) {
  const int few = pick_row_splits(M, N, K);
  if (few > 1 || M < TQ_BM || N % 16 || K % 128 || K < 1024) return few;
  const int64_t rows = (M + TQ_BM - 1) / TQ_BM, cols8 = (N + 255) / 256, cols4 = (N + 127) / 128,
                cols2 = (N + 63) / 64;
  if (K < 8192 && rows * cols2 * 4 < num_cus() * 3) return few;
  auto cost = [&](int S) {
    // in rounds of 256 x 256 tiles (103 us of K = 4096), of which 256 x 128 ones take 0.61 and 256 x 64 0.43
    auto full = [](int64_t tiles) { return (double)((tiles + num_cus() - 1) / num_cus()); };
    const int64_t tiles = rows * cols8 * S;
    const int pieces = quad_pieces(tiles, num_cus());
    const double wide = pieces == 1 ? full(tiles) : (double)(tiles / num_cus()) + (pieces == 2 ? 0.61 : 0.36);
    const double rounds = fmin(wide, fmin(full(rows * cols4 * S) * 0.61, full(rows * cols2 * S) * 0.43));
    return rounds * 103.0 / 4096 * K / S + (S - 1) * (double)M * N * 8 / 5e6;
  };
  return rows * cols8 * 2 <= num_cus() && cost(2) < 0.95 * cost(1) ? 2 : 1;
}

template <bool W8, int MODE>
void launch_tiled(const void* x, const void* W, const void* scales, int64_t M, int N, int K,
                  const Epilogue& epi, hipStream_t s) {
  // Up to 64 rows (a short prompt, a small batch held row-major): one sweep of the
  // weight-streaming kernel, which reads its activation fragments from the row-major matrix.
  // No tile kernel comes near it there (64 x 12288 x 4096, fp16: 101 us on 128 x 128 tiles).
  if (M <= 64)
    return launch_stream<W8, MODE, true>(x, W, scales, nullptr, 1, (int)M, N, K, epi, s, 0);
  // int8 weights, up to 256 rows: a sweep per 64 rows.  The int8 tile kernels need thousands of
  // rows to fill the chip (128 x 9216 x 9216: 303 us on 128 x 128 tiles, 51 us per sweep).
  if constexpr (W8) {
    if (M <= 256) {
      for (int64_t m0 = 0; m0 < M; m0 += 64)
        launch_stream<W8, MODE, true>(x, W, scales, nullptr, 1, (int)min((int64_t)64, M - m0), N,
                                      K, epi, s, m0);
      return;
    }
  }
  // int8: the 256 x 256 kernel once it fills the chip; the 128 x 128 one for the shapes in between
  const int64_t big_tiles = ((M + TB_BM - 1) / TB_BM) * ((N + TB_BN - 1) / TB_BN);
  if constexpr (!W8) {
    const TileForm f = tile_form(M, N, K, num_cus());
    if (f.kind == MSA_TILES_QUEUE)
      return launch_queue_rows<MODE>(x, W, nullptr, 1, (int)M, N, K, f.queue, epi, s);
    if (f.kind == MSA_TILES_EVEN) return launch_quad_plan<MODE, false>(x, W, M, N, K, 1, f.even, epi, nullptr, s);
    if (f.kind == MSA_TILES_WHOLE) {
      if (f.wf == 8) return launch_quad<MODE, 8>(x, W, scales, M, f.main, N, K, f.pieces, epi, s);
      if (f.wf == 4) return launch_quad<MODE, 4>(x, W, scales, M, f.main, N, K, 1, epi, s);
      return launch_quad<MODE, 2>(x, W, scales, M, f.main, N, K, 1, epi, s);
    }
    if (f.kind == MSA_TILES_FEW) {
      if (f.wf == 4) return launch_few_rows<MODE, 4, 4>(x, W, M, N, K, epi, s);
      if (f.rf == 4) return launch_few_rows<MODE, 8, 4>(x, W, M, N, K, epi, s);
      if (f.rf == 5) return launch_few_rows<MODE, 8, 5>(x, W, M, N, K, epi, s);
      if (f.rf == 6) return launch_few_rows<MODE, 8, 6>(x, W, M, N, K, epi, s);
      if (f.rf == 7) return launch_few_rows<MODE, 8, 7>(x, W, M, N, K, epi, s);
      return launch_few_rows<MODE, 8, 8>(x, W, M, N, K, epi, s);
    }
  }
  if constexpr (W8) if (K % (2 * TB_BK) == 0 && big_tiles >= num_cus()) {
    static std::atomic<uint64_t> lds_allowed{0};  // one mask per instantiation
    if (!allow_lds((const void*)linear_tiled_big_kernel<MODE>, TB_LDS_BYTES, lds_allowed))
      return;  // the launch check below reports the error
    // A ragged bottom block would cost a full extra round of workgroups for a few rows (a
    // prompt of 2^k tokens plus the leading end-of-sentence token always has one): up to 128
    // leftover rows go through the weight-streaming kernel instead, 64 rows at a time.
    int64_t M_main = M;
    const int64_t rem = M % TB_BM;
    if (rem > 0 && rem <= 128 && M > rem) M_main = M - rem;
    const dim3 grid((N + TB_BN - 1) / TB_BN, (unsigned)((M_main + TB_BM - 1) / TB_BM));
    hipLaunchKernelGGL((linear_tiled_big_kernel<MODE>), grid, dim3(TB_THREADS), TB_LDS_BYTES,
                       s, (const half_t*)x, W, (const half_t*)scales, M_main, N, K, epi);
    for (int64_t m0 = M_main; m0 < M; m0 += 64)
      launch_stream<W8, MODE, true>(x, W, scales, nullptr, 1, (int)min((int64_t)64, M - m0), N, K,
                                    epi, s, m0);
    return;
  }
  const dim3 grid((N + TL_BN - 1) / TL_BN, (unsigned)((M + TL_BM - 1) / TL_BM));
  hipLaunchKernelGGL((linear_tiled_kernel<W8, MODE>), grid, dim3(TL_THREADS), 0, s,
                     (const half_t*)x, W, (const half_t*)scales, M, N, K, epi);
}

template <int MODE>
void run_linear(const void* x, const void* W, const Epilogue& e, int64_t M, int N, int K,
                unsigned flags, hipStream_t s) {
  if (flags & MSA_IN_PACKED)
    launch_stream<false, MODE>(x, W, nullptr, nullptr, 1, (int)M, N, K, e, s);
  else
    launch_tiled<false, MODE>(x, W, nullptr, M, N, K, e, s);
}

int check_linear_args(const char* name, const void* x, const void* W, const void* y, int64_t M,
                      int N, int K, bool w8, unsigned flags, unsigned allowed) {
  MSA_REQUIRE(x && W && y, MSA_ERR_INVALID_ARG, "%s: null pointer", name);
  MSA_REQUIRE(M >= 0 && M < (1ll << 31) && N > 0 && K > 0, MSA_ERR_INVALID_ARG,
              "%s: bad shape M=%lld N=%d K=%d", name, (long long)M, N, K);
  MSA_REQUIRE(K % (w8 ? 64 : 32) == 0 && N % 16 == 0, MSA_ERR_INVALID_ARG,
              "%s: K=%d must be a multiple of %d and N=%d a multiple of 16", name, K, w8 ? 64 : 32,
              N);
  MSA_REQUIRE((M + TL_BM - 1) / TL_BM <= 65535, MSA_ERR_INVALID_ARG, "%s: M=%lld too large", name,
              (long long)M);
  MSA_REQUIRE((flags & ~allowed) == 0, MSA_ERR_INVALID_ARG, "%s: unsupported flags 0x%x", name,
              flags);
  MSA_REQUIRE(!(flags & (MSA_IN_PACKED | MSA_OUT_PACKED)) || M <= MSA_PACKED_MAX_ROWS,
              MSA_ERR_INVALID_ARG, "%s: packed activations exist only for M <= %d (M=%lld)", name,
              MSA_PACKED_MAX_ROWS, (long long)M);
  return MSA_OK;
}

// Split count that minimises what one workgroup moves through its L1: its weight tiles over
// its K range, the activation fragments of that K range once per tile group, and its fp32
// partial sums (written here, read back by the LayerNorm tail).  More splits mean more tiles
// per workgroup over a shorter K range, i.e. fewer activation bytes per weight byte.  At most `most` slices.
// In the queue kernel activations, which come from L2, cost half of as many weights, and a tile's sums more than the bytes they
// leave as: eight waves' go through LDS behind the loop.  Fitted to 130 products of 40 to 128 rows with their tails (us = 5 +
// 0.0278 per KB of weights + 0.0126 per KB of activations + 0.18 per 16 x 16 sums + 0.14 per 1000 of slices x columns, to 4.5 %);
// The shared-activation kernel in one pass, of nine to twelve tiles, has its waves' sums added by two, not eight: fp16, 128 rows with
// their tails, us, in two slices of queues and in four of it, 12288 x 12288 71 and 66, x 49152 233 and 211, 9216 x 36864 154 and 145,
// 64 rows of 12288 x 49152 197 and 191, of 12288 x 12288 58 and 61; int8, 64 rows of 12288 x 49152 124 and 119, 128 rows 163 and 184.  What
// is picked is 0.3 % slower than the best of 1, 2, 4 and 8 slices on average over 190 products of 40 to 128 rows.
int pick_splits(int64_t M, int N, int K, int wbytes, int most = 8) {
  if (M < 1 || M > MSA_PACKED_MAX_ROWS || N % 16 || K % 64) return 1;
  const bool w8 = wbytes == 1;
  const int MB = packed_row_blocks(M), ntiles = N / 16, nks = K / 32;
  // elsewhere: tiles that share one sweep over the activations (int8 has a 2 x 6 x 3 shape of the
  // shared-activation kernel for up to 18), and K steps per stage of the workgroup
  const int NT = MB > 2 ? (w8 && MB <= 4 ? SH_GROUP_W8 : SH_GROUP) : ST_NT;
  const int cus = num_cus();
  auto tiles = [&](int S) { return (ntiles + cus / S - 1) / (cus / S); };
  auto cost = [&](int S, bool queue) {
    const int tpw = tiles(S), groups = (tpw + NT - 1) / NT, rows = queue_rows((int)M);
    const double Ks = (double)K / S, w = tpw * 16.0 * Ks * wbytes, x = rows * 16.0 * Ks * 2, part = 5.1 * S * N;
    if (MB > 2 && queue) return w + 0.45 * x + 6500.0 * tpw * rows + part;
    if (MB > 2 && tpw <= SH_GROUP && (MB <= 4 || !w8)) return 1.05 * w + 0.45 * x + 3000.0 * tpw * rows + part + 80000.0;
    const double c = queue ? w + 0.45 * x + 6500.0 * tpw * rows + part : w + groups * MB * 16.0 * Ks * 2 + 2.0 * tpw * 16 * M * 4;
    return c * (MB > 2 ? 2 : 1) * (1.0 + 0.02 * S);  // ties go to fewer splits; of more rows, this is what is left
  };
  // Up to 32 rows fewer slices than the stream kernel would take only in queues: its waves' chains would be as much longer (fp16, 32
  // rows of 5120 x 5120, fp32 sums off by 1.09e-7 in four slices, in two by 1.32e-7; and 15.9 us with the tail in queues, 16.3).
  // More than it would take only in queues, too: int8, 9 rows of 6640 x 8256, four 15.9 us, eight 19.7.
  int best = 1, least = 1;
  if (MB <= 2)
    for (int S = 2; S <= most && S <= cus && nks / S >= ST_KG * 4; S *= 2)
      if (cost(S, false) < cost(least, false)) least = S;
  double best_cost = 0;
  for (int S = 1; S <= most && S <= cus; S *= 2) {
    const bool queue = queue_takes((int)M, w8, tiles(S));
    const int stage = !queue ? (MB > 2 ? 16 : ST_KG * 4) : MB > 2 ? 8 * (w8 ? 2 : 1) : ST_KG * 4;
    if (nks / S < stage) break;  // every wave needs a full stage of K steps
    if (!queue && MB <= 2 && S != least) continue;
    const double c = cost(S, queue);
    if (best_cost == 0 || c < best_cost) best = S, best_cost = c;
  }
  return best;
}

}  // namespace
