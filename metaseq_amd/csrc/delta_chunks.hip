// The gated delta rule over segments of many tokens, sixteen tokens at a time on the fp32 matrix cores.
//
// With S0 the state in front of a chunk, p_i the decays of tokens 1 .. i multiplied (per key channel), and
// k'_i = p_i k_i, q'_i = p_i q_i, the recurrence S_i = g_i S_{i-1} + k_i u_i^T,
// u_i = beta_i (v_i - (g_i S_{i-1})^T k_i), o_i = S_i^T q_i of recurrent.hip's scan is
//   U = T (V - K' S0),     T = (I + L)^{-1} diag(beta),  L_ij = beta_i k_i . (p_i / p_j) k_j   (j < i),
//   O = Q' S0 + A U,       A_ij = q_i . (p_i / p_j) k_j                                          (j <= i),
//   S = p_C S0 + K^^T U,   k^_j = (p_C / p_j) k_j.
// No quotient of decays is ever formed: p_i / p_j is the product of the decays between the two tokens,
// multiplied up token by token, so a channel that forgets at once is as exact as in the scan.  All of
// it is fp32, the products on v_mfma_f32_16x16x4_f32.
//
// Two kernels.  What does not depend on S0 (T, A, the norms of k and q; for few segments with decays per channel also
// K', Q' and K^) is computed for all chunks of all heads at once, a wave each, and left in a scratch record; then the
// chunks of a (segment, head, some columns) are walked one after the other.  A scan step's chain of LDS reads, two
// dots, a sum over lanes and the update takes 500 cycles per token whatever the machine has idle; a
// chunk's chain takes 2900 per sixteen with one decay per head and 2400 with decays per channel
// where few segments leave a workgroup a CU of its own.  Where many fill the chip the matrix cores are the bound: 104
// fp32 products of 32 cycles per wave and chunk, two such waves per SIMD, 6650 cycles of the 11000 a chunk takes.
// Measured, both kernels against the scan, 32 heads of 128 x 128: one segment of 1500 tokens 128 us against 349
// (decays per channel 123 against 351), 8 x 1024 tokens 322 against 788 (362 against 1003).
#include <math.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "attention_tiles.h"
#include "common.h"

namespace {

constexpr int DC_TOK = 16;
constexpr int DC_WIDE = 128;  // workgroups of several column tiles from which on they take over
constexpr int DC_READY = 512;  // workgroups of one column tile up to which ready operands are the faster
constexpr int64_t DC_LONG = 40 << 20;  // floats of long records kept at a time
// A record: T and A (16 x 16, row-major), then per token the factors that are one number for all channels.
// The norms are divided out in two steps.  Operands are multiplied by a power of two (SK of k, SQ of q), which is exact
// and brings them near unit length, so that no product overflows that the scan's unit vectors would not; a vector whose
// squared norm overflows has the factor 0, as in the scan.  The rest, between 1 and 2, the loops below apply to 16 x 16
// results: of K' S0 (1 / |k|), Q' S0 (scale / |q|) and U (1 / |k|), each times the token's product of decays where a
// head has one decay, and that product over the chunk.  Past the segment's end the factors are 0.
constexpr int DC_T = 0, DC_A = 256, DC_FK = 512, DC_FQ = 528, DC_FU = 544, DC_GC = 560, DC_SK = 576, DC_SQ = 592,
              DC_REC = 608;
// For few segments with decays per channel a record goes on with K', Q' and K^ (16 x DP each) in the order in which the
// lanes of the MFMAs take them, 1 KB per 16 channels, and p_C.
template <int DP, bool READY>
constexpr int rec_floats = DC_REC + (READY ? 3 * DC_TOK * DP + DP : 0);
// (DC_GC holds sixteen copies: one address for all lanes would be a scalar load, whose latency every LDS
// barrier waits for)

__device__ __forceinline__ bool finite(float v) { return fabsf(v) <= 3.4028234663852886e38f; }

// records of a segment start here: chunks are counted from each segment's own start, and
// ceil(n / 16) <= floor((first + n) / 16) - floor(first / 16) + 1
__device__ __forceinline__ int64_t record_of(int first, int seg, int chunk, int heads, int h, int floats) {
  return ((int64_t)(first / DC_TOK + seg + chunk) * heads + h) * floats;
}
// Long records are kept for `count` chunks of every segment at a time, from chunk `from` on (count 0: for all chunks, as
// above): a launch sees that portion as the segment.  False: nothing of the segment lies in it.
struct Portion {
  int from, count;
  __device__ __forceinline__ bool narrow(int& first, int& n, int& pos) const {
    if (count == 0) return true;
    if (from > 0) {
      if (pos < 0 || n <= from * DC_TOK) return false;
      first += from * DC_TOK;
      n -= from * DC_TOK;
      pos = 1;  // (behind tokens: the state goes on)
    }
    if (pos >= 0) n = min(n, count * DC_TOK);
    return true;
  }
  __device__ __forceinline__ int64_t record(int first, int seg, int chunk, int heads, int h, int floats) const {
    return count == 0 ? record_of(first, seg, chunk, heads, h, floats)
                      : ((int64_t)(seg * count + chunk) * heads + h) * floats;
  }
};

template <int N, int... I, class F>
__device__ __forceinline__ void each(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void each(F&& f) {  // f(0) .. f(N - 1), the number a constant
  each<N>(f, std::make_integer_sequence<int, N>{});
}

// Sums of 64 values over the 64 lanes, two lanes' worth at a time: the lane keeps one half of the values and
// gives the other half away, so that 64 sums take 63 additions and not 64 x 6.  Lane l ends with the
// sum of value l.
__device__ __forceinline__ float transposed_sums(float (&v)[64], int lane) {
#pragma unroll
  for (int t = 0; t < 32; ++t) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, v[t]),
                                                    __builtin_bit_cast(unsigned, v[t + 32]), false, false);
    v[t] = __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
  }
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, v[t]),
                                                    __builtin_bit_cast(unsigned, v[t + 16]), false, false);
    v[t] = __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
  }
#define DC_HALVE(W, CTRL)                                    \
  _Pragma("unroll") for (int t = 0; t < W; ++t) {            \
    const bool up = lane & W;                                \
    const float keep = up ? v[t + W] : v[t], give = up ? v[t] : v[t + W]; \
    v[t] = keep + dpp_move<CTRL, 0xf>(0.f, give);            \
  }
  DC_HALVE(8, 0x128)  // row_ror:8
  DC_HALVE(4, 0x141)  // row_half_mirror: the lane with the other bits 0 .. 2
  DC_HALVE(2, 0x4E)   // quad_perm [2,3,0,1]
  DC_HALVE(1, 0xB1)   // quad_perm [1,0,3,2]
#undef DC_HALVE
  return v[0];
}

// Place of a sum in the order the loops below form them: per token j first q_j . k_j, then for every later token i
// the sums of L_ij and A_ij.
constexpr int sum_at(int j) { return 32 * j - j * j; }
constexpr int DC_SUMS = sum_at(DC_TOK);  // 256
static_assert(DC_SUMS % 64 == 0, "whole groups of sums");

// One wave per (chunk, head).  Bound: the vector ALU (for 128 channels some 800 multiply-adds and
// 700 steps of the sums per chunk and lane).  The decays between two tokens are multiplied up as j's row moves from token to token.
template <typename T, int DP, bool CH, bool READY>
__global__ __launch_bounds__(256) void delta_prepare_kernel(
    const T* __restrict__ qkv, int64_t ld, const float* __restrict__ ba, int ldba,
    const float* __restrict__ decay_rate, const float* __restrict__ dt_bias,
    const float* __restrict__ decay, int heads, int kv_heads, float q_scale, float* __restrict__ records,
    const int32_t* __restrict__ seg_start, const int32_t* __restrict__ seg_pos, Portion portion) {
  static_assert(CH || !READY, "records of whole operands are for decays per channel");
  constexpr int CE = (DP + 63) / 64;  // channels per lane
  __shared__ float sums[4][DC_SUMS], tok[4][6][DC_TOK];  // tok: beta, rest of 1 / |k| and of scale / |q|, decay, SK, SQ
  const int s = blockIdx.z, t0 = blockIdx.x * DC_TOK;
  int first = seg_start[s], n = seg_start[s + 1] - first, pos = seg_pos[s];
  if (READY && !portion.narrow(first, n, pos)) return;
  if (t0 >= n || pos < 0) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int h_own = blockIdx.y * 4 + wave, h = min(h_own, heads - 1);
  const int hk = h / (heads / kv_heads), c0 = lane * CE;
  const bool live = c0 < DP;
  const T* base = qkv + (int64_t)first * ld + hk * DP + (live ? c0 : 0);
  float k[DC_TOK][CE], q[DC_TOK][CE], g[CH ? DC_TOK : 1][CE];
#pragma unroll
  for (int t = 0; t < DC_TOK; ++t) {
    const int tt = min(t0 + t, n - 1);
    const bool use = live && t0 + t < n;
    const T* p = base + (int64_t)tt * ld;
#pragma unroll
    for (int e = 0; e < CE; ++e) {
      const float qv = (float)p[e], kv = (float)p[kv_heads * DP + e];
      q[t][e] = use ? qv : 0.f;
      k[t][e] = use ? kv : 0.f;
      if constexpr (CH) {
        const float d = decay[((int64_t)(first + tt) * heads + h) * DP + (live ? c0 : 0) + e];
        g[t][e] = use ? d : 1.f;
      }
    }
  }
  auto dot = [&](const float (&a)[CE], const float (&b)[CE]) {
    float d = a[0] * b[0];
#pragma unroll
    for (int e = 1; e < CE; ++e) d = fmaf(a[e], b[e], d);
    return d;
  };
  float v[64];
#pragma unroll
  for (int t = 0; t < DC_TOK; ++t) {
    v[t] = dot(k[t], k[t]);
    v[DC_TOK + t] = dot(q[t], q[t]);
    v[2 * DC_TOK + t] = v[3 * DC_TOK + t] = 0.f;
  }
  const float square = transposed_sums(v, lane);  // of k (lanes 0 .. 15) or q (16 .. 31)
  if (lane < 2 * DC_TOK) {
    // (the few factors per token in 64 bits: one rounding each, and no time that shows beside the sums)
    const int t = lane & 15;
    const bool of_q = lane >> 4, in = t0 + t < n;
    const double norm = sqrt((double)square + 1e-6), scale = of_q ? q_scale : 1.f;
    int e = 0;
    const double rest = isfinite(norm) ? frexp(norm, &e) : norm;
    tok[wave][of_q ? 5 : 4][t] = in && isfinite(norm) ? ldexpf(1.f, -e) : 0.f;
    tok[wave][of_q ? 2 : 1][t] = in ? (float)(scale / rest) : 0.f;
  }
  if (lane < DC_TOK) {
    const bool in = t0 + lane < n;
    const float* z = ba + (int64_t)(first + min(t0 + lane, n - 1)) * ldba;
    tok[wave][0][lane] = in ? (float)(1.0 / (1.0 + exp(-(double)z[h]))) : 0.f;
    if (!CH) tok[wave][3][lane] = in ? decay_of(z[heads + h] + dt_bias[h], decay_rate[h]) : 1.f;
  }
  __syncthreads();
  float gs[CH ? 1 : DC_TOK];
  if constexpr (!CH) {
#pragma unroll
    for (int t = 0; t < DC_TOK; ++t) gs[t] = tok[wave][3][t];
  }
#pragma unroll
  for (int t = 0; t < DC_TOK; ++t)
#pragma unroll
    for (int e = 0; e < CE; ++e) {
      k[t][e] *= tok[wave][4][t];
      q[t][e] *= tok[wave][5][t];
    }
  auto emit = [&](auto at, float x) {
    constexpr int A = decltype(at)::value;
    v[A & 63] = x;
    if constexpr ((A & 63) == 63) sums[wave][A - 63 + lane] = transposed_sums(v, lane);
  };
  each<DC_TOK>([&](auto jc) {
    constexpr int j = decltype(jc)::value, at = sum_at(j);
    emit(std::integral_constant<int, at>{}, dot(q[j], k[j]));
    float w[CE];
#pragma unroll
    for (int e = 0; e < CE; ++e) w[e] = k[j][e];
    each<DC_TOK - 1 - j>([&](auto ic) {
      constexpr int i = j + 1 + decltype(ic)::value;
#pragma unroll
      for (int e = 0; e < CE; ++e) w[e] *= CH ? g[CH ? i : 0][e] : gs[CH ? 0 : i];
      emit(std::integral_constant<int, at + 2 * (i - j) - 1>{}, dot(k[i], w));
      emit(std::integral_constant<int, at + 2 * (i - j)>{}, dot(q[i], w));
    });
  });
  __syncthreads();
  const float* sm = sums[wave];
  constexpr int REC = rec_floats<DP, READY>;
  float* rec = records + (READY ? portion.record(first, s, blockIdx.x, heads, h, REC)
                                : record_of(first, s, blockIdx.x, heads, h, REC));
  if constexpr (READY) {
    // K' and Q' go through LDS (rows padded: the lanes that write a token lie 68 floats apart), so that the stores
    // are whole lines; a channel's K^ is 16 bytes of four tokens as it lies.  75 MB for 1500 tokens of 32 heads:
    // 23 -> 39 us.
    constexpr int TILES = DP / 16, PITCH = 68;
    __shared__ float turn[4][TILES * 4 * PITCH];
    float* tw = turn[wave];
    float p[CE];
    auto turned = [&](const float (&x)[DC_TOK][CE], float* to) {
#pragma unroll
      for (int e = 0; e < CE; ++e) p[e] = 1.f;
#pragma unroll
      for (int t = 0; t < DC_TOK; ++t)
#pragma unroll
        for (int e = 0; e < CE; ++e) {
          p[e] *= g[t][e];
          const int c = c0 + e;
          if (live) tw[(c >> 2) * PITCH + t * 4 + (c & 3)] = x[t][e] * p[e];
        }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < TILES; ++i) {
        const float4_t v = *reinterpret_cast<const float4_t*>(tw + (i * 4 + (lane >> 4)) * PITCH + (lane & 15) * 4);
        if (h_own < heads) *reinterpret_cast<float4_t*>(to + i * 256 + lane * 4) = v;
      }
      __syncthreads();
    };
    turned(k, rec + DC_REC);
    turned(q, rec + DC_REC + DC_TOK * DP);
    if (h_own < heads && live) {
#pragma unroll
      for (int e = 0; e < CE; ++e) {
        const int c = c0 + e;
        float* to = rec + DC_REC + 2 * DC_TOK * DP + (c >> 4) * 256 + (c & 15) * 4;
        float m = 1.f, late = 1.f, x[DC_TOK];
#pragma unroll
        for (int t = DC_TOK / 2; t < DC_TOK; ++t) late *= g[t][e];
#pragma unroll
        for (int t = DC_TOK - 1; t >= 0; --t) {
          if (t == DC_TOK / 2 - 1) m = late;
          x[t] = k[t][e] * m;
          m *= g[t][e];
        }
#pragma unroll
        for (int t = 0; t < DC_TOK; t += 4)
          *reinterpret_cast<float4_t*>(to + t * 16) = float4_t{x[t], x[t + 1], x[t + 2], x[t + 3]};
        rec[DC_REC + 3 * DC_TOK * DP + c] = p[e];
      }
    }
  }
  if (h_own >= heads) return;
  const float *beta = tok[wave][0], *fk = tok[wave][1], *fq = tok[wave][2];
  if (lane < DC_TOK) {  // column `lane` of T, by substitution
    float x[DC_TOK];
    each<DC_TOK>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      float d = 0.f;
#pragma unroll
      for (int j = 0; j < i; ++j) d = fmaf(sm[sum_at(j) + 2 * (i - j) - 1] * fk[j], x[j], d);
      x[i] = i < lane ? 0.f : beta[i] * ((i == lane ? 1.f : 0.f) - fk[i] * d);
      rec[DC_T + i * DC_TOK + lane] = x[i];
    });
    // A row of T that is not finite (a beta, decay or key that is not) would reach the chunk's earlier tokens as a U
    // that is 0 x NaN in A U.  Its factor of K' S0 says so: right_hand_side() takes every column out from there on.
    int bad = DC_TOK;
#pragma unroll
    for (int i = DC_TOK - 1; i >= 0; --i)
      if (!finite(x[i])) bad = i;
#pragma unroll
    for (int d = 1; d < DC_TOK; d *= 2) bad = min(bad, __shfl_xor(bad, d, MSA_WAVE));
    float before = 1.f, after = 1.f;
    if constexpr (!CH) {
#pragma unroll
      for (int i = 0; i < DC_TOK; ++i) (i <= lane ? before : after) *= gs[i];
      rec[DC_GC + lane] = before * after;
    }
    rec[DC_FK + lane] = lane == bad ? __builtin_nanf("") : fk[lane] * before;
    rec[DC_FQ + lane] = fq[lane] * before;
    rec[DC_FU + lane] = fk[lane] * after;
    rec[DC_SK + lane] = tok[wave][4][lane];
    rec[DC_SQ + lane] = tok[wave][5][lane];
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int i = (lane >> 4) * 4 + e, j = lane & 15;
    const float raw = sm[i >= j ? sum_at(j) + 2 * (i - j) : 0];
    rec[DC_A + i * DC_TOK + j] = i >= j ? fq[i] * fk[j] * raw : 0.f;
  }
}

// What the chunk loops read of a chunk, twice: one is staged while the other is in use.  With one decay
// per head K' and K^ are both k, the decays being factors of the results.
template <int DP, bool CH>
struct Operands {
  static constexpr int KS = DP + 4;   // a row stride that keeps 16-byte reads free of conflicts
  float k[2][DC_TOK][KS], q[2][DC_TOK][KS];  // K', Q'
  float kh[CH ? 2 : 1][CH ? DC_TOK : 1][CH ? KS : 4];  // K^
  float gc[CH ? 2 : 1][CH ? DP : 4];         // p_C
  // element (token 4 lg + r, row) of K^ for r = 0 .. 3: the A operand of the state's update
  __device__ __forceinline__ float4_t key_column(int b, int lg, int row) const {
    float4_t v;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = CH ? kh[CH ? b : 0][CH ? lg * 4 + r : 0][CH ? row : 0] : k[b][lg * 4 + r][row];
    return v;
  }
};

// The four staging waves of a workgroup (thread t of 256).  One decay per head: a thread moves 8 channels of a
// token.  Decays per channel: a thread owns two channels of k (the first two waves) or q over half of
// the chunk's tokens and multiplies the decays up; the lane 32 away has the other half.
// Chunks are requested two ahead.  The loops of these kernels take chunks in pairs and without conditions
// around their loads, so that each wait is for the oldest chunk alone; an odd number of chunks is made even
// by one past the end, whose k, q and U are set to 0 and its decays to 1, which changes nothing.
template <typename T, int DP, bool CH>
struct Stager {
  typedef T t4 __attribute__((ext_vector_type(4), aligned(8)));
  typedef T t2 __attribute__((ext_vector_type(2), aligned(2 * sizeof(T))));
  typedef float f2 __attribute__((ext_vector_type(2), aligned(8)));
  struct Raw {
    t4 x[CH ? 1 : 4];       // one decay per head: 8 of k, 8 of q
    t2 y[CH ? 8 : 1];
    f2 g[CH ? 8 : 1];
    float f[CH ? 8 : 2];    // SK or SQ of the thread's tokens; one decay per head: SK and SQ of its token
  };
  const T *ksrc, *qsrc;      // uniform: the head's first channel of the segment's first token
  const float *dsrc, *fsrc;
  int64_t ld, ldd, ldf;
  int n, t, half;
  unsigned at;               // first channel of the thread
  bool is_k, live;

  __device__ Stager(int t_, const T* rows, int64_t ld_, const float* decay, int first, int heads, int kv_heads,
                    int h, int n_, const float* rec0) {
    t = t_;
    n = n_;
    ld = ld_;
    const int hk = h / (heads / kv_heads);
    qsrc = rows + hk * DP;
    ksrc = qsrc + kv_heads * DP;
    ldd = (int64_t)heads * DP;
    dsrc = CH ? decay + ((int64_t)first * heads + h) * DP : nullptr;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    is_k = wave < 2;
    half = (t >> 5) & 1;
    const int pair = (wave & 1) * 32 + (t & 31);
    live = CH ? pair < DP / 2 : t < 2 * DP;
    at = CH ? min(pair, DP / 2 - 1) * 2 : min(t, 2 * DP - 1) % (DP / 8) * 8;
    ldf = (int64_t)heads * DC_REC;
    fsrc = rec0 + (CH ? (is_k ? DC_SK : DC_SQ) + half * 8 : DC_SK + min(t, 2 * DP - 1) / (DP / 8));
  }
  __device__ __forceinline__ void fetch(Raw& a, int c) const {
    const float* fac = fsrc + min(c, (n - 1) / DC_TOK) * ldf;
    if constexpr (CH) {
#pragma unroll
      for (int i = 0; i < 8; i += 4) {
        const float4_t f = *reinterpret_cast<const float4_t*>(fac + i);
#pragma unroll
        for (int j = 0; j < 4; ++j) a.f[CH ? i + j : 0] = f[j];
      }
      const T* src = is_k ? ksrc : qsrc;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int tt = min(c * DC_TOK + half * 8 + i, n - 1);
        a.y[i] = *reinterpret_cast<const t2*>(src + tt * ld + at);
        a.g[i] = *reinterpret_cast<const f2*>(dsrc + tt * ldd + at);
      }
    } else {
      const int64_t row = min(c * DC_TOK + min(t, 2 * DP - 1) / (DP / 8), n - 1) * ld + at;
      a.x[0] = *reinterpret_cast<const t4*>(ksrc + row);
      a.x[1] = *reinterpret_cast<const t4*>(ksrc + row + 4);
      a.x[2] = *reinterpret_cast<const t4*>(qsrc + row);
      a.x[3] = *reinterpret_cast<const t4*>(qsrc + row + 4);
      a.f[0] = fac[0];
      a.f[1] = fac[DC_SQ - DC_SK];
    }
  }
  __device__ __forceinline__ void stage(Operands<DP, CH>& L, const Raw& a, int c) const {
    const int b = c & 1;
    const bool past = c * DC_TOK >= n;
    if constexpr (!CH) {
      if (!live) return;
      const int tok = t / (DP / 8);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float f = past ? 0.f : a.f[i >> 1];
        *reinterpret_cast<float4_t*>(&(i < 2 ? L.k : L.q)[b][tok][at + (i & 1) * 4]) =
            float4_t{(float)a.x[i][0], (float)a.x[i][1], (float)a.x[i][2], (float)a.x[i][3]} * f;
      }
      return;
    }
    f2 g[8], p = {1.f, 1.f};
    const int left = n - c * DC_TOK - half * 8;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      g[i] = a.g[CH ? i : 0];
      if (i >= left) g[i] = f2{1.f, 1.f};
      p[0] *= g[i][0], p[1] *= g[i][1];
    }
    const f2 other = {__shfl_xor(p[0], 32, MSA_WAVE), __shfl_xor(p[1], 32, MSA_WAVE)};
    if (!live) return;
    const int tok = half * 8;
    f2 m = {half ? other[0] : 1.f, half ? other[1] : 1.f};
    f2 x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      x[i] = f2{(float)a.y[CH ? i : 0][0], (float)a.y[CH ? i : 0][1]} * (past ? 0.f : a.f[CH ? i : 0]);
      m[0] *= g[i][0], m[1] *= g[i][1];
      *reinterpret_cast<f2*>(&(is_k ? L.k : L.q)[b][tok + i][at]) = f2{x[i][0] * m[0], x[i][1] * m[1]};
    }
    if (is_k) {
      m = f2{half ? 1.f : other[0], half ? 1.f : other[1]};
#pragma unroll
      for (int i = 7; i >= 0; --i) {
        *reinterpret_cast<f2*>(&L.kh[CH ? b : 0][CH ? tok + i : 0][CH ? at : 0]) = f2{x[i][0] * m[0], x[i][1] * m[1]};
        m[0] *= g[i][0], m[1] *= g[i][1];
      }
    } else if (half) {
      *reinterpret_cast<f2*>(&L.gc[CH ? b : 0][CH ? at : 0]) = m;
    }
  }
};

__device__ __forceinline__ float4_t mfma4(float4_t a, float4_t b, float4_t c) {  // c + a (16 x 16) b (16 x 16)
#pragma unroll
  for (int r = 0; r < 4; ++r) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], c, 0, 0, 0);
  return c;
}
// c[t] += a[t] b[t] for N independent accumulators, in turn
template <int N>
__device__ __forceinline__ void mfma4(const float4_t (&a)[N], const float4_t (&b)[N], float4_t (&c)[N]) {
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int t = 0; t < N; ++t) c[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t][r], b[t][r], c[t], 0, 0, 0);
}
// The new state: what a chunk adds is summed by itself, so that the state is rounded once per chunk.  Error of
// outputs and state against 64 bits, 1000 tokens, heads of 128: 2.9e-7 and 4.3e-8 (the scan: 3.2e-7 and 5.3e-8),
// with decays per channel 1.6e-7 and 2.3e-8 (2.8e-7 and 5.1e-8); summed onto the decayed state 2.9e-7 and 5.2e-8.
__device__ __forceinline__ float4_t decayed_plus(float4_t s, float4_t g, float4_t add) {
#pragma unroll
  for (int r = 0; r < 4; ++r) s[r] = fmaf(s[r], g[r], add[r]);
  return s;
}

// A lane's part of a record: tokens 4 lg .., and row lm of T
struct Factors {
  float4_t t, k, q, u;
  float gc;
  __device__ __forceinline__ void fetch(const float* rec0, int64_t rec_step, int c, int nch, int lm, int lg, bool ch) {
    const float* rec = rec0 + min(c, nch - 1) * rec_step;
    t = *reinterpret_cast<const float4_t*>(rec + DC_T + lm * DC_TOK + lg * 4);
    k = *reinterpret_cast<const float4_t*>(rec + DC_FK + lg * 4);
    q = *reinterpret_cast<const float4_t*>(rec + DC_FQ + lg * 4);
    u = *reinterpret_cast<const float4_t*>(rec + DC_FU + lg * 4);
    gc = ch ? 1.f : rec[DC_GC + lm];
  }
  // U on its way to the state; a chunk past the end changes nothing, whatever its U is
  __device__ __forceinline__ void finish(float4_t& x, int bad, int lg, int c, int nch) {
    if (c >= nch) gc = 1.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = c >= nch ? 0.f : lg * 4 + r >= bad ? __builtin_nanf("") : x[r] * u[r];
  }
};

// V - K' S0 of a lane's four tokens 4 lg .. of one column.  A value that is not finite would reach the
// earlier tokens of its chunk as 0 x NaN: such a column goes through U with zeros from that token on
// (returned; 16: all are finite) and gets NaN there afterwards.
template <typename T>
__device__ __forceinline__ int right_hand_side(const T (&v)[4], float4_t ks, float4_t f, int lg, float4_t& out) {
  bool fine = true;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    out[r] = fmaf(-f[r], ks[r], (float)v[r]);
    fine &= finite(out[r]);
  }
  int bad = DC_TOK;
  if (!__all(fine)) {  // uniform
#pragma unroll
    for (int r = 3; r >= 0; --r)
      if (!finite(out[r])) bad = lg * 4 + r;
    bad = min(bad, __shfl_xor(bad, 16, MSA_WAVE));
    bad = min(bad, __shfl_xor(bad, 32, MSA_WAVE));
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (lg * 4 + r >= bad) out[r] = 0.f;
  }
  return bad;
}

template <int DP, bool CH>
struct StagedLds {
  Operands<DP, CH> op;
  float a[4][DC_TOK][DC_TOK + 4];            // A of the chunk being staged, used and finished
  float4_t ks[4][64], qs[2][4][64], u[2][64];
  int bad[2][16];
};

// Few segments: a workgroup owns one segment, one head and 16 of its columns for all of the segment's chunks.
// Waves 0 .. 3 hold the state, a quarter of its rows each, as MFMA accumulators (a lane: four rows of one
// column), which are the B operands of the next chunk's products as they lie; they sum K' S0 through
// LDS, form U redundantly and update their rows.  Waves 4 .. 7 run beside them, between the two barriers of a chunk:
// they finish the previous chunk's outputs and stage the next chunk (before the first barrier, beside the short
// product K' S0, 1500 tokens took 124 us, here 115).
template <typename T, int DP, bool CH>
__global__ __launch_bounds__(512) void delta_chunk_kernel(
    const T* __restrict__ qkv, int64_t ld, const float* __restrict__ decay, int heads, int kv_heads, int vp,
    float* __restrict__ state, const float* __restrict__ records, float* __restrict__ o,
    const int32_t* __restrict__ seg_start, const int32_t* __restrict__ seg_slot,
    const int32_t* __restrict__ seg_pos) {
  constexpr int TILES = DP / 16, TPW = (TILES + 3) / 4;  // 16-row tiles of the state, per wave
  extern __shared__ __attribute__((aligned(16))) char dc_lds[];
  StagedLds<DP, CH>& L = *reinterpret_cast<StagedLds<DP, CH>*>(dc_lds);
  const int s = blockIdx.z, h = blockIdx.y, col0 = blockIdx.x * 16;
  const int first = seg_start[s], n = seg_start[s + 1] - first, pos = seg_pos[s];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lm = lane & 15, lg = lane >> 4;
  float* out = o + (int64_t)first * heads * vp + h * vp + col0;
  if (pos < 0) {
    for (int i = tid; i < n * 16; i += 512) out[(int64_t)(i >> 4) * heads * vp + (i & 15)] = 0.f;
    return;
  }
  if (n <= 0) return empty_segment(state + (((int64_t)seg_slot[s] * heads + h) * vp + col0) * DP, 16 * DP, pos);
  const int nch = (n + DC_TOK - 1) / DC_TOK;
  const T* rows = qkv + (int64_t)first * ld;
  const float* rec0 = records + record_of(first, s, 0, heads, h, DC_REC);
  const int64_t rec_step = (int64_t)heads * DC_REC;

  if (wave < 4) {
    const int v_at = 2 * kv_heads * DP + h * vp + col0 + lm;
    float* st = state + (((int64_t)seg_slot[s] * heads + h) * vp + col0 + lm) * DP + lg * 4;
    float4_t S[TPW];
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      S[t] = float4_t{0.f, 0.f, 0.f, 0.f};
      if (pos > 0 && wave * TPW + t < TILES)
        S[t] = *reinterpret_cast<const float4_t*>(st + (wave * TPW + t) * 16);
    }
    struct Ahead {
      T v[4];
      Factors f;
    } ahead[2];
    auto fetch = [&](Ahead& a, int c) {
#pragma unroll
      for (int r = 0; r < 4; ++r) a.v[r] = rows[(int64_t)min(c * DC_TOK + lg * 4 + r, n - 1) * ld + v_at];
      a.f.fetch(rec0, rec_step, c, nch, lm, lg, CH);
    };
    auto chunk = [&](Ahead& a, int c) {
      const int b = c & 1;
      auto times_state = [&](const float* x) {
        // (tiles past the end: a state of zeros times some row in bounds)
        float4_t sum[TPW], a[TPW];
#pragma unroll
        for (int t = 0; t < TPW; ++t) {
          sum[t] = float4_t{0.f, 0.f, 0.f, 0.f};
          a[t] = *reinterpret_cast<const float4_t*>(x + min(wave * TPW + t, TILES - 1) * 16);
        }
        mfma4(a, S, sum);
#pragma unroll
        for (int t = 1; t < TPW; ++t) sum[0] += sum[t];
        return sum[0];
      };
      L.ks[wave][lane] = times_state(&L.op.k[b][lm][lg * 4]);
      lds_barrier();  // A
      float4_t ks = L.ks[0][lane];
#pragma unroll
      for (int w = 1; w < 4; ++w) ks += L.ks[w][lane];
      L.qs[b][wave][lane] = times_state(&L.op.q[b][lm][lg * 4]) * a.f.q;
      float4_t rhs;
      const int bad = right_hand_side(a.v, ks, a.f.k, lg, rhs);
      float4_t u = mfma4(a.f.t, rhs, float4_t{0.f, 0.f, 0.f, 0.f});
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (lg * 4 + r >= bad) u[r] = 0.f;
      if (wave == 0) {
        L.u[b][lane] = u;
        if (lane < 16) L.bad[b][lane] = bad;
      }
      a.f.finish(u, bad, lg, c, nch);
      const float gc = a.f.gc;
      fetch(a, c + 2);
      float4_t kh[TPW], us[TPW], g[TPW], add[TPW];
#pragma unroll
      for (int t = 0; t < TPW; ++t) {
        const int row = min(wave * TPW + t, TILES - 1) * 16;
        if constexpr (CH) g[t] = *reinterpret_cast<const float4_t*>(&L.op.gc[CH ? b : 0][CH ? row + lg * 4 : 0]);
        else g[t] = float4_t{gc, gc, gc, gc};
        add[t] = float4_t{0.f, 0.f, 0.f, 0.f};
        kh[t] = L.op.key_column(b, lg, row + lm);
        us[t] = u;
        if (wave * TPW + t >= TILES) kh[t] = us[t] = float4_t{0.f, 0.f, 0.f, 0.f};
      }
      mfma4(kh, us, add);
#pragma unroll
      for (int t = 0; t < TPW; ++t) S[t] = decayed_plus(S[t], g[t], add[t]);
      lds_barrier();  // B
    };
    fetch(ahead[0], 0);
    fetch(ahead[1], 1);
    lds_barrier();  // chunk 0 is staged
    for (int c = 0; c < nch; c += 2) {
      chunk(ahead[0], c);
      chunk(ahead[1], c + 1);
    }
#pragma unroll
    for (int t = 0; t < TPW; ++t)
      if (wave * TPW + t < TILES) *reinterpret_cast<float4_t*>(st + (wave * TPW + t) * 16) = S[t];
    return;
  }

  typedef Stager<T, DP, CH> St;
  const int ht = tid - 256;
  const St stager(ht, rows, ld, decay, first, heads, kv_heads, h, n, rec0);
  struct Raw {
    typename St::Raw r;
    float a;  // element ht of A
  } raw[2];
  auto fetch = [&](Raw& x, int c) {
    stager.fetch(x.r, c);
    x.a = rec0[min(c, nch - 1) * rec_step + DC_A + ht];
  };
  auto stage = [&](const Raw& x, int c) {
    L.a[c & 3][ht >> 4][ht & 15] = x.a;
    stager.stage(L.op, x.r, c);
  };
  // outputs of chunk c, by one of the four waves in turn (with decays per channel, of the two that stage q)
  auto finish = [&](int c) {
    if (c < 0 || (CH ? (c & 1) != wave - 6 : (c & 3) != wave - 4)) return;
    const int b = c & 1;
    float4_t y = L.qs[b][0][lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) y += L.qs[b][w][lane];
    y = mfma4(*reinterpret_cast<const float4_t*>(&L.a[c & 3][lm][lg * 4]), L.u[b][lane], y);
    const int bad = L.bad[b][lm];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = c * DC_TOK + lg * 4 + r;
      if (t < n) out[(int64_t)t * heads * vp + lm] = lg * 4 + r >= bad ? __builtin_nanf("") : y[r];
    }
  };
  fetch(raw[0], 0);
  fetch(raw[1], 1);
  stage(raw[0], 0);
  fetch(raw[0], 2);
  lds_barrier();
  auto beside = [&](Raw& x, int c) {  // x holds chunk c + 1
    lds_barrier();  // A
    finish(c - 1);
    stage(x, c + 1);
    fetch(x, c + 3);
    lds_barrier();  // B
  };
  for (int c = 0; c < nch; c += 2) {
    beside(raw[1], c);
    beside(raw[0], c + 1);
  }
  finish((nch + 1) / 2 * 2 - 1);  // (the loop finished all chunks before that one)
}

struct ReadyLds {
  float4_t ks[2][4][64], qs[2][4][64], u[2][64];
  int bad[2][16];
};

// The same for decays per channel, which would be multiplied up again for every 16 columns: K', Q' and K^ come from the
// chunk's record straight into the state waves' registers, two chunks ahead; the workgroups of a head run on one
// XCD and share its L2 lines.  Waves 4 .. 7 finish the outputs, a chunk each in turn.  One barrier per chunk, behind
// its K' S0: what the waves hand each other is double buffered.  Both kernels, 32 heads of 128, one segment of 128 / 512 /
// 1500 / 16384 tokens: 25 / 50 / 123 / 1333 us (staged 29 / 67 / 176 / 1820).  With one decay per head staging is a copy,
// and the longer records cost more than they save (128 / 512 tokens 23.8 / 51.0 us staged, 25.7 / 53.7 so; 16 heads of 128 x
// 96, 8 x 512 tokens 117 and 134).
template <typename T, int DP>
__global__ __launch_bounds__(512) void delta_chunk_ready_kernel(
    const T* __restrict__ qkv, int64_t ld, int heads, int kv_heads, int vp,
    float* __restrict__ state, const float* __restrict__ records, float* __restrict__ o,
    const int32_t* __restrict__ seg_start, const int32_t* __restrict__ seg_slot,
    const int32_t* __restrict__ seg_pos, Portion portion) {
  constexpr int TILES = DP / 16, TPW = (TILES + 3) / 4;  // 16-row tiles of the state, per wave
  constexpr int REC = rec_floats<DP, true>;
  __shared__ ReadyLds L;
  const int s = blockIdx.z, h = blockIdx.x, col0 = blockIdx.y * 16;
  int first = seg_start[s], n = seg_start[s + 1] - first, pos = seg_pos[s];
  if (!portion.narrow(first, n, pos)) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lm = lane & 15, lg = lane >> 4;
  float* out = o + (int64_t)first * heads * vp + h * vp + col0;
  if (pos < 0) {
    for (int i = tid; i < n * 16; i += 512) out[(int64_t)(i >> 4) * heads * vp + (i & 15)] = 0.f;
    return;
  }
  if (n <= 0) return empty_segment(state + (((int64_t)seg_slot[s] * heads + h) * vp + col0) * DP, 16 * DP, pos);
  const int nch = (n + DC_TOK - 1) / DC_TOK;
  const T* rows = qkv + (int64_t)first * ld;
  const float* rec0 = records + portion.record(first, s, 0, heads, h, REC);
  const int64_t rec_step = (int64_t)heads * REC;

  if (wave < 4) {
    const int v_at = 2 * kv_heads * DP + h * vp + col0 + lm;
    float* st = state + (((int64_t)seg_slot[s] * heads + h) * vp + col0 + lm) * DP + lg * 4;
    float4_t S[TPW];
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      S[t] = float4_t{0.f, 0.f, 0.f, 0.f};
      if (pos > 0 && wave * TPW + t < TILES)
        S[t] = *reinterpret_cast<const float4_t*>(st + (wave * TPW + t) * 16);
    }
    struct Ahead {
      float4_t k[TPW], q[TPW], kh[TPW], g[TPW];
      T v[4];
      Factors f;
    } ahead[2];
    // (chunks past the end: the last one again, of which no result is used)
    auto fetch = [&](Ahead& a, int c) {
      const float* ready = rec0 + min(c, nch - 1) * rec_step + DC_REC;
#pragma unroll
      for (int t = 0; t < TPW; ++t) {
        const int tile = min(wave * TPW + t, TILES - 1);  // past the end: a state of zeros times some tile in bounds
        a.k[t] = *reinterpret_cast<const float4_t*>(ready + tile * 256 + lane * 4);
        a.q[t] = *reinterpret_cast<const float4_t*>(ready + DC_TOK * DP + tile * 256 + lane * 4);
        a.kh[t] = *reinterpret_cast<const float4_t*>(ready + 2 * DC_TOK * DP + tile * 256 + lane * 4);
        a.g[t] = *reinterpret_cast<const float4_t*>(ready + 3 * DC_TOK * DP + tile * 16 + lg * 4);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) a.v[r] = rows[(int64_t)min(c * DC_TOK + lg * 4 + r, n - 1) * ld + v_at];
      a.f.fetch(rec0, rec_step, c, nch, lm, lg, true);
    };
    auto times_state = [&](const float4_t (&x)[TPW]) {
      float4_t sum[TPW];
#pragma unroll
      for (int t = 0; t < TPW; ++t) sum[t] = float4_t{0.f, 0.f, 0.f, 0.f};
      mfma4(x, S, sum);
#pragma unroll
      for (int t = 1; t < TPW; ++t) sum[0] += sum[t];
      return sum[0];
    };
    auto chunk = [&](Ahead& a, const Ahead& next, int c) {
      const int b = c & 1;
      float4_t part[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) part[w] = L.ks[b][w][lane];
      const float4_t y = times_state(a.q) * a.f.q;
      float4_t ks = part[0];
#pragma unroll
      for (int w = 1; w < 4; ++w) ks += part[w];
      float4_t rhs;
      const int bad = right_hand_side(a.v, ks, a.f.k, lg, rhs);
      float4_t u = mfma4(a.f.t, rhs, float4_t{0.f, 0.f, 0.f, 0.f});
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (lg * 4 + r >= bad) u[r] = 0.f;
      L.qs[b][wave][lane] = y;
      if (wave == 0) {
        L.u[b][lane] = u;
        if (lane < 16) L.bad[b][lane] = bad;
      }
      a.f.finish(u, bad, lg, c, nch);
      float4_t us[TPW], add[TPW];
#pragma unroll
      for (int t = 0; t < TPW; ++t) {
        add[t] = float4_t{0.f, 0.f, 0.f, 0.f};
        us[t] = u;
        if (wave * TPW + t >= TILES) a.kh[t] = us[t] = float4_t{0.f, 0.f, 0.f, 0.f};
      }
      mfma4(a.kh, us, add);
#pragma unroll
      for (int t = 0; t < TPW; ++t) S[t] = decayed_plus(S[t], a.g[t], add[t]);
      fetch(a, c + 2);
      L.ks[b ^ 1][wave][lane] = times_state(next.k);
      lds_barrier();
    };
    fetch(ahead[0], 0);
    fetch(ahead[1], 1);
    L.ks[0][wave][lane] = times_state(ahead[0].k);
    lds_barrier();
    int c = 0;
    for (; c + 1 < nch; c += 2) {
      chunk(ahead[0], ahead[1], c);
      chunk(ahead[1], ahead[0], c + 1);
    }
    if (c < nch) chunk(ahead[0], ahead[1], c);
#pragma unroll
    for (int t = 0; t < TPW; ++t)
      if (wave * TPW + t < TILES) *reinterpret_cast<float4_t*>(st + (wave * TPW + t) * 16) = S[t];
    return;
  }

  // outputs of chunk c, whose sums lie in LDS behind the barrier of chunk c + 1
  const float* rec_a = rec0 + DC_A + lm * DC_TOK + lg * 4;
  const int turn = wave - 4;
  float4_t a = *reinterpret_cast<const float4_t*>(rec_a + min(turn, nch - 1) * rec_step);
  lds_barrier();
  for (int c = 0; c < nch; ++c) {
    lds_barrier();
    if ((c & 3) != turn) continue;
    const int b = c & 1;
    float4_t y = L.qs[b][0][lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) y += L.qs[b][w][lane];
    y = mfma4(a, L.u[b][lane], y);
    const int bad = L.bad[b][lm];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = c * DC_TOK + lg * 4 + r;
      if (t < n) out[(int64_t)t * heads * vp + lm] = lg * 4 + r >= bad ? __builtin_nanf("") : y[r];
    }
    a = *reinterpret_cast<const float4_t*>(rec_a + min(c + 4, nch - 1) * rec_step);
  }
}

// Many segments: a workgroup owns CT x 16 columns of a head, one wave 16 of them with all rows of the state, so
// that nothing is summed between waves and k, q and decays are staged for CT column tiles at once; four
// more waves stage.  One barrier per chunk.
// CHAINS: accumulators of K' S0 and Q' S0.  Two are enough to keep the matrix cores busy; widths with a last partial
// group, which few segments' kernels would take otherwise, get one per tile of the state as there (error of the outputs
// against 64 bits, 8 x 300 tokens, 16 heads of 96 columns: two 1.76e-7, one per tile 1.58e-7 as staged; 208 and 211 us).
template <typename T, int DP, bool CH, int CT, int CHAINS>
__global__ __launch_bounds__((CT + 4) * 64) void delta_chunk_wide_kernel(
    const T* __restrict__ qkv, int64_t ld, const float* __restrict__ decay, int heads, int kv_heads, int vp,
    float* __restrict__ state, const float* __restrict__ records, float* __restrict__ o,
    const int32_t* __restrict__ seg_start, const int32_t* __restrict__ seg_slot,
    const int32_t* __restrict__ seg_pos) {
  constexpr int TILES = DP / 16;
  extern __shared__ __attribute__((aligned(16))) char dc_lds[];
  Operands<DP, CH>& L = *reinterpret_cast<Operands<DP, CH>*>(dc_lds);
  const int s = blockIdx.z, h = blockIdx.y, col0 = blockIdx.x * (CT * 16);
  const int first = seg_start[s], n = seg_start[s + 1] - first, pos = seg_pos[s];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lm = lane & 15, lg = lane >> 4;
  const int cols = min(CT * 16, vp - col0);  // the last group of a width that is not whole groups has fewer
  if (pos < 0) {
    for (int i = tid; i < n * CT * 16; i += (CT + 4) * 64)
      if (i % (CT * 16) < cols)
        o[(int64_t)(first + i / (CT * 16)) * heads * vp + h * vp + col0 + i % (CT * 16)] = 0.f;
    return;
  }
  if (n <= 0) return empty_segment(state + (((int64_t)seg_slot[s] * heads + h) * vp + col0) * DP, cols * DP, pos);
  const int nch = (n + DC_TOK - 1) / DC_TOK;
  const T* rows = qkv + (int64_t)first * ld;
  const float* rec0 = records + record_of(first, s, 0, heads, h, DC_REC);
  const int64_t rec_step = (int64_t)heads * DC_REC;
  if (wave >= CT) {
    typedef Stager<T, DP, CH> St;
    const St stager(tid - CT * 64, rows, ld, decay, first, heads, kv_heads, h, n, rec0);
    typename St::Raw raw[2];
    stager.fetch(raw[0], 0);
    stager.fetch(raw[1], 1);
    stager.stage(L, raw[0], 0);
    stager.fetch(raw[0], 2);
    lds_barrier();
    auto beside = [&](typename St::Raw& x, int c) {
      stager.stage(L, x, c + 1);  // (past the last chunk: copies of the last row times 0)
      stager.fetch(x, c + 3);
      lds_barrier();
    };
    for (int c = 0; c < nch; c += 2) {
      beside(raw[1], c);
      beside(raw[0], c + 1);
    }
    return;
  }
  if (wave * 16 >= cols) {  // no columns: the barriers of the others
    lds_barrier();
    for (int c = 0; c < nch; c += 2) {
      lds_barrier();
      lds_barrier();
    }
    return;
  }
  const int col = col0 + wave * 16 + lm;
  const T* vsrc = rows + 2 * kv_heads * DP + h * vp + col;
  float* out = o + (int64_t)first * heads * vp + h * vp + col;
  float* st = state + (((int64_t)seg_slot[s] * heads + h) * vp + col) * DP + lg * 4;
  float4_t S[TILES];
#pragma unroll
  for (int t = 0; t < TILES; ++t) {
    S[t] = float4_t{0.f, 0.f, 0.f, 0.f};
    if (pos > 0) S[t] = *reinterpret_cast<const float4_t*>(st + t * 16);
  }
  struct Ahead {
    T v[4];
    float4_t a;
    Factors f;
  } ahead[2];
  auto fetch = [&](Ahead& x, int c) {
#pragma unroll
    for (int r = 0; r < 4; ++r) x.v[r] = vsrc[(int64_t)min(c * DC_TOK + lg * 4 + r, n - 1) * ld];
    x.f.fetch(rec0, rec_step, c, nch, lm, lg, CH);
    x.a = *reinterpret_cast<const float4_t*>(rec0 + min(c, nch - 1) * rec_step + DC_A + lm * DC_TOK + lg * 4);
  };
  auto chunk = [&](Ahead& x, int c) {
    const int b = c & 1;
    auto times_state = [&](const float* p) {
      float4_t sum[CHAINS];
#pragma unroll
      for (int i = 0; i < CHAINS; ++i) sum[i] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < TILES; t += CHAINS) {
        float4_t a[CHAINS], x[CHAINS];
#pragma unroll
        for (int i = 0; i < CHAINS; ++i) {
          a[i] = *reinterpret_cast<const float4_t*>(p + (t + i) * 16);
          x[i] = S[t + i];
        }
        mfma4(a, x, sum);
      }
#pragma unroll
      for (int i = 0; i < CHAINS; i += 2) {
        if (i + 1 < CHAINS) sum[i] += sum[i + 1];
        if (i > 0) sum[0] += sum[i];
      }
      return sum[0];
    };
    const float4_t ks = times_state(&L.k[b][lm][lg * 4]);
    float4_t y = times_state(&L.q[b][lm][lg * 4]) * x.f.q;
    float4_t rhs;
    const int bad = right_hand_side(x.v, ks, x.f.k, lg, rhs);
    float4_t u = mfma4(x.f.t, rhs, float4_t{0.f, 0.f, 0.f, 0.f});
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (lg * 4 + r >= bad) u[r] = 0.f;
    y = mfma4(x.a, u, y);
    x.f.finish(u, bad, lg, c, nch);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (lg * 4 + r >= bad) y[r] = __builtin_nanf("");
    const float gc = x.f.gc;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = c * DC_TOK + lg * 4 + r;
      if (t < n) out[(int64_t)t * heads * vp] = y[r];
    }
    fetch(x, c + 2);
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      float4_t g = {gc, gc, gc, gc};
      if constexpr (CH) g = *reinterpret_cast<const float4_t*>(&L.gc[CH ? b : 0][CH ? t * 16 + lg * 4 : 0]);
      S[t] = decayed_plus(S[t], g, mfma4(L.key_column(b, lg, t * 16 + lm), u, float4_t{0.f, 0.f, 0.f, 0.f}));
    }
    lds_barrier();
  };
  fetch(ahead[0], 0);
  fetch(ahead[1], 1);
  lds_barrier();
  for (int c = 0; c < nch; c += 2) {
    chunk(ahead[0], c);
    chunk(ahead[1], c + 1);
  }
#pragma unroll
  for (int t = 0; t < TILES; ++t) *reinterpret_cast<float4_t*>(st + t * 16) = S[t];
}

// Which kernel walks the chunks: wide workgroups of 64 or 128 columns, or sixteen columns each (few segments), the operands
// staged from the rows or ready in the records.  Ready ones spare every column tile the staging, which with decays per
// channel is most of the work, until their 27 KB per chunk and head are what is waited for: then the wide kernel, whose
// staging serves four tiles, is the better one for any width, and a single tile stages for itself.  128 keys, decays per
// channel, us staged / ready / wide of 64, 1000 tokens of one segment: 64 heads of 96 columns (384 workgroups) 236 / 158 /
// 186, 96 of 80 (480) 245 / 185 / 196, 128 of 48 (384) 254 / 215 / 201, 128 of 80 (640) 358 / 277 / 211; 500 tokens, 256 of
// 32 (512) 153 / 165 / 127; 8 x 1024 tokens, 16 of 96 (768) 359 / 285 / 211; one tile, 128 heads 150 / 148 / 199, 256 heads
// 195 / 268 / 239.
enum Form { STAGED, READY, WIDE_64, WIDE_128, WIDE_ANY, FORMS };
Form form_of(const msa_delta_args& a, const msa_batch* b) {
  const int64_t units = (int64_t)b->nseg * a.heads;
  if (a.vp % 128 == 0 && units >= DC_WIDE) return WIDE_128;
  if (a.vp % 64 == 0 && units * (a.vp / 64) >= DC_WIDE) return WIDE_64;
  if (!a.decay) return STAGED;
  if (a.vp == 16) return units <= DC_WIDE ? READY : STAGED;
  return a.vp % 64 != 0 && units * (a.vp / 16) >= DC_READY ? WIDE_ANY : READY;
}

// Chunks of every segment whose long records are kept at a time, all portions alike; 0: all.  32 heads of 128, one segment
// of 4096 / 16384 tokens: all at once (226 and 903 MB) 355 / 1368 us, in portions of 64 / 32 / 16 / 8 Mi floats - / 1420, 333 /
// 1332, 342 / 1447, 405 / 1635: up to some 160 MB the records are still in the memory-side cache when they are read,
// and a portion costs two launches and the loads in front of its first chunk.
int portion_chunks(const msa_delta_args& a, const msa_batch* b) {
  const int64_t layer = (int64_t)a.heads * (DC_REC + (3 * DC_TOK + 1) * a.dp);
  if (((int64_t)b->M / DC_TOK + b->nseg) * layer <= DC_LONG) return 0;
  const int chunks = (b->max_count + DC_TOK - 1) / DC_TOK;
  const int most = (int)std::max<int64_t>(1, DC_LONG / (layer * b->nseg));
  const int portions = (chunks + most - 1) / most;
  return (chunks + portions - 1) / portions;
}

template <typename T, int DP, bool CH>
int run_chunks(const msa_delta_args& a, const msa_batch* b, float* scratch, hipStream_t s) {
  const int chunks = (b->max_count + DC_TOK - 1) / DC_TOK;
  const Form form = form_of(a, b);
  auto prepare = [&](auto kernel, int count, Portion p) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)count, (a.heads + 3) / 4, b->nseg), dim3(256), 0, s, (const T*)a.qkv,
                       a.ld, a.ba, a.ldba, a.decay_rate, a.dt_bias, a.decay, a.heads, a.kv_heads,
                       (float)pow((double)a.dim, -0.5), scratch, b->seg_start, b->seg_pos, p);
  };
  if constexpr (CH) {
    if (form == READY) {
      const int at_once = portion_chunks(a, b), step = at_once > 0 ? at_once : chunks;
      for (int from = 0; from < chunks; from += step) {
        const Portion p{from, at_once};
        prepare(delta_prepare_kernel<T, DP, CH, true>, std::min(step, chunks - from), p);
        hipLaunchKernelGGL((delta_chunk_ready_kernel<T, DP>), dim3(a.heads, a.vp / 16, b->nseg), dim3(512), 0, s,
                           (const T*)a.qkv, a.ld, a.heads, a.kv_heads, a.vp, a.state, scratch, a.o, b->seg_start,
                           b->seg_slot, b->seg_pos, p);
      }
      return MSA_OK;
    }
  }
  prepare(delta_prepare_kernel<T, DP, CH, false>, chunks, Portion{});
  auto kernel = form == WIDE_128  ? delta_chunk_wide_kernel<T, DP, CH, 8, 2>
                : form == WIDE_64 ? delta_chunk_wide_kernel<T, DP, CH, 4, 2>
                                  : delta_chunk_kernel<T, DP, CH>;
  if constexpr (CH) {
    if (form == WIDE_ANY) kernel = delta_chunk_wide_kernel<T, DP, CH, 4, DP / 16>;
  }
  const int cols = form == WIDE_128 ? 128 : form == STAGED ? 16 : 64;
  const int threads = form == WIDE_128 ? 768 : 512;
  const int bytes = form == STAGED ? (int)sizeof(StagedLds<DP, CH>) : (int)sizeof(Operands<DP, CH>);
  static std::atomic<uint64_t> raised[FORMS];
  if (!raise_lds((const void*)kernel, bytes, raised[form])) {
    msa_set_error("msa_delta_scan_chunks: %d bytes of LDS refused", bytes);
    return MSA_ERR_HIP;
  }
  hipLaunchKernelGGL(kernel, dim3((a.vp + cols - 1) / cols, a.heads, b->nseg), dim3(threads), bytes, s,
                     (const T*)a.qkv, a.ld, a.decay, a.heads, a.kv_heads, a.vp, a.state, scratch, a.o, b->seg_start,
                     b->seg_slot, b->seg_pos);
  return MSA_OK;
}

template <typename T>
int pick_chunks(const msa_delta_args& a, const msa_batch* b, float* scratch, hipStream_t s) {
#define DC_CASE(DP) \
  case DP:          \
    return a.decay ? run_chunks<T, DP, true>(a, b, scratch, s) : run_chunks<T, DP, false>(a, b, scratch, s);
  switch (a.dp) {
    DC_CASE(32)
    DC_CASE(64)
    DC_CASE(96)
    DC_CASE(128)
  }
#undef DC_CASE
  return MSA_ERR_INVALID_ARG;  // not reached: msa_delta_scratch_floats is 0 for other sizes
}

}  // namespace

// The scan stays faster for few short segments (both kernels cost some 15 us before the first token; one segment of
// 96 / 112 / 128 tokens: 22.2 / 23.9 / 23.8 us against 25.5 / 28.6 / 31.5, with decays per channel 22.5 / 23.7 /
// 25.0 against 25.1 / 30.1 / 34.2; of 64 tokens 17.9 and 17.2 by the scan); where the segments fill the chip the chunks
// win from the first length tried (8 x 48 tokens 32 us against 44, seven segments of 20 and one of 64 32 against 36).
constexpr int DC_FROM = 96, DC_FROM_WIDE = 48;

extern "C" int64_t msa_delta_scratch_floats(const msa_delta_args* a, const msa_batch* b) {
  if (!a || !b || a->heads <= 0 || a->dp > 128) return 0;
  if (b->max_count < ((int64_t)b->nseg * a->heads >= DC_WIDE ? DC_FROM_WIDE : DC_FROM)) return 0;
  const int64_t all = ((int64_t)b->M / DC_TOK + b->nseg) * a->heads, staged = all * DC_REC;
  // (a caller that has not set vp gets enough for any)
  if (!a->decay || (a->vp > 0 && form_of(*a, b) != READY)) return staged;
  const int at_once = portion_chunks(*a, b);
  const int64_t ready = (at_once > 0 ? (int64_t)at_once * b->nseg * a->heads : all) * (DC_REC + (3 * DC_TOK + 1) * a->dp);
  return a->vp > 0 ? ready : std::max(ready, staged);
}

int msa_launch_delta_chunks(const msa_delta_args& a, const msa_batch* b, float* scratch, hipStream_t s) {
  return a.dtype == MSA_BF16 ? pick_chunks<bf16_t>(a, b, scratch, s) : pick_chunks<float>(a, b, scratch, s);
}
