#pragma once
// The queue kernels: products of packed rows, 33 .. 128 of them or fewer with many tiles to a workgroup, and of 129 .. 256
// row-major rows (gemm_kernels.h chooses).
#include "gemm_kernels.h"

namespace {

// ---- queue kernel (33 .. 128 packed rows; fewer where the workgroup has five to nine tiles) ----
// Bound: what a CU receives, weights from HBM and activations from L2.  A probe that only loads (KB of either per wave, by
// direct loads to LDS) gets 27 GB/s per CU of weights alone (7.0 TB/s over the chip), 25 of them beside as many bytes of activations
// (6.3 TB/s) and 16 beside three times as many, with 16 KB in flight or more; the shared-activation kernel, whose waves meet at a
// barrier per stage and wait for the next stage's activations in order behind a stage of weights, got 16 in the first case.
//
// Here no wave waits for another: the KL waves are K lanes, every one with all NT tiles and MB row blocks, and each has a
// queue of its own in LDS that direct loads fill (R slots of one K step: NT KB of weights, then MB KB of activations; an int8
// slot covers two steps).  A slot is read into registers, requested anew, and then multiplied.  Every activation
// still comes to the CU once.  Two waves per SIMD where the sums and a slot fit 256 registers, one where they do not.  The
// waves' sums are added through LDS in fixed order, as many tiles at a time as fit, and all waves take part in the epilogue.
// Up to two row blocks take half or a quarter of the slices here that the stream kernel would take (pick_splits): a wave's sums
// are set aside up to four times on its way, so that none is a longer chain than that kernel's.  fp32 sums, off by (stream kernel's
// slices / fewer, one chain / set aside): int8 32 x 9216 x 36864 1.74e-7 / 2.28 / 1.39, fp16 24 x 5120 x 20480 1.42 / 1.76 / 1.27, 32 x
// 12288 x 12288 1.45 / 1.89 / 1.27; 0.1 to 0.6 us (with its tail the first 62.0 and 62.5, the second 37.0 and 37.2).
//
// us, shared-activation kernel and this: fp16 57 x 16384 x 4096 33.3 and 26.9, 57 x 12288 x 4096 23.7 and 21.5, 64 x 20480 x 5120
// 47.9 and 38.0, 64 x 36864 x 9216 114 and 104, 64 x 3072 x 768 7.7 and 5.1, 72 x 16384 x 4096 35 and 28.1, 104 rows 35.3 and
// 33.0, 128 rows 38 and 35, 128 x 3072 x 768 12.5 and 6.3, 128 x 8192 x 2048 22 and 14.5; int8 64 x 36864 x 9216 75 and 65.6, 64 x
// 27648 x 9216 65 and 53, 72 x 36864 x 9216 126 and 70, 104 rows 127 and 87, 128 x 27648 x 9216 102 and 76.  Against the
// stream kernel: int8 32 x 9216 x 36864 in four slices 74.5 and 56, 8 x 36864 x 9216 60 and 54; fp16 32 x 5120 x 20480 in four
// slices 39.9 and 33.3.
// Other numbers of waves (57 x 16384 x 4096): 4 28.4, 6 27.1, 10 27.4, 12 28.7, 16 31.4.
template <int MB, bool W8, int NT>
struct QueueCfg {
  static constexpr int STEPS = W8 ? 2 : 1;       // 32-wide steps of a slot
  static constexpr int LOADS = STEPS * MB + NT;  // of 1 KB each
  static constexpr int SLOT = LOADS * 1024;
  static constexpr bool ASIDE = MB <= 2;  // slices' sums are set aside after a quarter of the slots, of eight 32-wide steps at least
  // registers: sums, one slot's fragments, and some for addresses and the expansion of int8
  static constexpr int REGS = 4 * ((ASIDE ? 2 : 1) * MB * NT + LOADS) + (W8 ? 20 : 8);
  static constexpr int KL = REGS <= 256 && 8 * SLOT <= 160 * 1024 ? 8 : 4;
  static constexpr int FIT = 160 * 1024 / (KL * SLOT), R = FIT > 4 ? 4 : FIT;
  static constexpr int JFIT = 160 * 1024 / (KL * MB * 1024), J = JFIT > NT ? NT : JFIT;  // tiles summed at a time
  static constexpr int RING = KL * R * SLOT, RED = KL * J * MB * 1024;
  static constexpr int LDS_BYTES = RING > RED ? RING : RED;
  static constexpr bool SUMS_FIT = 4 * MB * NT <= 256;  // one accumulator bank
  static_assert(R >= 1 && J >= 1, "a CU has 160 KB of LDS");
};

template <int OFF, bool ONCE>
__device__ __forceinline__ void queue_load(uint32_t vo, const char* sb, uint32_t m0) {
  if constexpr (ONCE)
    asm volatile("global_load_lds_dwordx4 %0, %1 offset:%2 nt" ::"v"(vo), "s"(sb), "n"(OFF), "{m0}"(m0) : "memory");
  else
    asm volatile("global_load_lds_dwordx4 %0, %1 offset:%2" ::"v"(vo), "s"(sb), "n"(OFF), "{m0}"(m0) : "memory");
}

// mbl: row blocks of the packed activations (MB of them hold rows)
template <int MB, bool W8, int MODE, int NT>
__global__ __launch_bounds__((QueueCfg<MB, W8, NT>::KL * 64)) void linear_queue_kernel(
    const half_t* __restrict__ xp, const void* __restrict__ Wp, const half_t* __restrict__ scales,
    float* __restrict__ part, int M, int N, int K, int tiles_per_wg, int ks_per_split, int mbl, Epilogue epi) {
  using C = QueueCfg<MB, W8, NT>;
  constexpr int STEPS = C::STEPS, R = C::R, L = C::LOADS, KL = C::KL;
  extern __shared__ __attribute__((aligned(16))) char lds_queue[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t lane_off = (uint32_t)lane * 16u;
  const int ntiles = N >> 4, nblk = (K >> 5) / STEPS;
  const int tile_begin = blockIdx.x * tiles_per_wg;
  const int tile_end = min(ntiles, tile_begin + tiles_per_wg);
  const int b_begin = blockIdx.y * (ks_per_split / STEPS);
  const int b_end = min(nblk, b_begin + ks_per_split / STEPS);
  // the wave's slots: blocks b_begin + wave + KL i
  const int n = b_begin + wave < b_end ? (b_end - b_begin - wave + KL - 1) / KL : 0;

  // Loads j .. j + 3 of a group share one M0; the instruction offset moves both addresses, so that the tiles' bases, which
  // do not follow one another in memory, are set back by it.  Tiles past the last one repeat it and are dropped at the end.
  const char* wb[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
    wb[j] = (const char*)Wp + (int64_t)min(tile_begin + j, tile_end - 1) * nblk * 1024 - (j % 4) * 1024;
  uint32_t sc[NT];  // int8: the row's fp16 scale
#pragma unroll
  for (int j = 0; j < NT; ++j)
    sc[j] = W8 ? reinterpret_cast<const uint16_t*>(scales)[min(tile_begin + j, tile_end - 1) * 16 + (lane & 15)] : 0u;
  const char* ring = lds_queue + wave * (R * C::SLOT);
  const uint32_t ring_at = (uint32_t)(uintptr_t)(tq_lds_void*)lds_queue + wave * (R * C::SLOT);
  auto request = [&](int slot, int i) {
    const uint32_t b = (uint32_t)(b_begin + wave + KL * i);
    const uint32_t at = ring_at + slot * C::SLOT;
    const uint32_t wv = lane_off + b * 1024u;
    tq_static_for<NT>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      queue_load<(j % 4) * 1024, true>(wv, wb[j], at + (j / 4) * 4096);
    });
    tq_static_for<STEPS>([&](auto uc) {
      constexpr int u = decltype(uc)::value;
      const uint32_t xv = lane_off + (b * STEPS + u) * ((uint32_t)mbl * 1024u);
      tq_static_for<MB>([&](auto fc) {
        constexpr int f = decltype(fc)::value;
        queue_load<(f % 4) * 1024, false>(xv + (f / 4) * 4096, (const char*)xp, at + (NT + u * MB) * 1024 + (f / 4) * 4096);
      });
    });
  };

  float4_t acc[NT][MB], aside[C::ASIDE ? NT : 1][MB];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[j][mb] = aside[C::ASIDE ? j : 0][mb] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (r < n) request(r, r);
  // (the scales are waited for here: at their first use the wait would cover the queue, step after step)
#pragma unroll
  for (int j = 0; j < NT; ++j)
    if (W8) asm volatile("" : "+v"(sc[j]));
  const int quarter = part ? max((n + 3) / 4, 8 / STEPS) : n + 1;  // (whole products have the stream kernel's chains)
  int slot = 0, until = quarter;
  for (int i = 0; i < n; ++i) {
    // loads complete in order: slot i is there when no more than those of the R - 1 slots behind it are on their way
    if (i + R - 1 < n)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((R - 1) * L) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const half8_t* from = reinterpret_cast<const half8_t*>(ring + slot * C::SLOT) + lane;
    half8_t w[NT], x[STEPS * MB];
#pragma unroll
    for (int j = 0; j < NT; ++j) w[j] = from[j * 64];
#pragma unroll
    for (int f = 0; f < STEPS * MB; ++f) x[f] = from[(NT + f) * 64];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read, before it is written again
    if (i + R < n) request(slot, i + R);
    slot = slot == R - 1 ? 0 : slot + 1;
#pragma unroll
    for (int u = 0; u < STEPS; ++u)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        half8_t a;
        if constexpr (W8) {
          typedef uint32_t u4 __attribute__((ext_vector_type(4)));
          const u4 raw = __builtin_bit_cast(u4, w[j]);
          const half_t scj = __builtin_bit_cast(half2_t, sc[j])[0];
          a = u ? dequant8(raw[2], raw[3], scj) : dequant8(raw[0], raw[1], scj);
        } else {
          a = w[j];
        }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[j][mb] = mfma_16x16x32<MODE>(a, x[u * MB + mb], acc[j][mb]);
      }
    if constexpr (C::ASIDE)
      if (--until == 0) {
        until = quarter;
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) aside[j][mb] += acc[j][mb], acc[j][mb] = float4_t{0.f, 0.f, 0.f, 0.f};
      }
  }
  if constexpr (C::ASIDE) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) acc[j][mb] += aside[j][mb];
  }

  // the waves' sums in wave order, J tiles at a time: [wave][tile][row block][lane]
  float4_t* red = reinterpret_cast<float4_t*>(lds_queue);
  constexpr int TOT = C::J * MB, PER = (TOT + KL - 1) / KL;  // pieces of 16 rows x 16 columns, of a wave
  // what the epilogue reads is requested in front of the reduction, where there are few pieces to a wave
  constexpr bool AHEAD = PER <= 4 && (!is_bf<MODE> || MODE == MODE_BF_POST);
#pragma unroll
  for (int j0 = 0; j0 < NT; j0 += C::J) {
    Ahead<MODE> ahead[AHEAD ? PER : 1];
    if (AHEAD && !part) {
#pragma unroll
      for (int q = 0; q < (AHEAD ? PER : 0); ++q) {
        const int p = min(wave + q * KL, TOT - 1);
        const int t = min(tile_begin + j0 + p / MB, tile_end - 1);
        ahead[q] = epilogue_ahead<MODE>(epi, min(p % MB * 16 + (lane & 15), M - 1), t * 16 + ((lane >> 4) << 2));
      }
    }
    __syncthreads();  // every wave is done with its queue, or with the sums before
#pragma unroll
    for (int j = j0; j < j0 + C::J && j < NT; ++j)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) red[((wave * C::J + j - j0) * MB + mb) * 64 + lane] = acc[j][mb];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int p = wave + q * KL, j = j0 + p / MB, mb = p % MB, t = tile_begin + j;
      if (p >= TOT || j >= NT || t >= tile_end) continue;
      float4_t sum = red[p * 64 + lane];
#pragma unroll
      for (int k = 1; k < KL; ++k) sum += red[(k * TOT + p) * 64 + lane];
      const int m = mb * 16 + (lane & 15), c = t * 16 + ((lane >> 4) << 2);
      if (m >= M) continue;
      if (part)
        *reinterpret_cast<float4_t*>(part + ((int64_t)blockIdx.y * M + m) * N + c) = sum;
      else
        epilogue4<MODE, AHEAD>(epi, m, c, sum, ahead[AHEAD ? q : 0]);
    }
  }
}

// ---- the same for 129 .. 256 row-major rows ----
// Two workgroups share a column of NT tiles, each with half of the rows (MB blocks of 16, the last row repeated), next to each
// other on one XCD, so that the weights come from HBM once.  A slot is 64 deep: a load takes a 128-byte line of each of eight
// rows, chunk c of row r at position c ^ (r / 2) % 8, as in the tile kernels, whose fragment reads then meet no bank conflicts;
// a tile's two 1 KB blocks follow each other in memory.
//
// The tile kernels' four waves wait for each other at every 32-wide step, and cut so few rows and columns into few tiles.  us,
// tiles and this, 129 / 200 / 256 rows: 3072 x 768 10.5 / 11.3 / 12.3 and 6.5 / 7.3 / 7.7; 6144 x 2048 18.4 / 20.3 / 22.6 and
// 12.6 / 15.4 / 16.5; 4096 x 4096 29.7 / 33.9 / 39.0 and 16.9 / 20.3 / 22.4; 8192 x 4096 32.3 / 36.2 / 41.0 and 24.5 / 28.5 /
// 31.2; 10240 x 2560 (five tiles) 24.3 / 26.7 / 30.6 and 19.8 / 24.2 / 26.1.  With six tiles or more a CU receives as many bytes as
// with 128 x 128 tiles, and its one wave per SIMD has no second slot to wait with: 12288 x 2048 22.5 / 23.2 / 25.0 and 19.7 / 24.8
// / 25.8, 200 x 16384 x 4096 42.6 and 49.
template <int MB, int NT>
struct QueueRowsCfg {
  static constexpr int LOADS = 2 * (MB + NT), SLOT = LOADS * 1024;
  static constexpr int REGS = 4 * (MB * NT + LOADS) + 40;
  static constexpr int KL = REGS <= 256 && 8 * SLOT <= 160 * 1024 ? 8 : 4;
  static constexpr int FIT = 160 * 1024 / (KL * SLOT), R = FIT > 4 ? 4 : FIT;
  static constexpr int JFIT = 160 * 1024 / (KL * MB * 1024), J = JFIT > NT ? NT : JFIT;
  static constexpr int RING = KL * R * SLOT, RED = KL * J * MB * 1024;
  static constexpr int LDS_BYTES = RING > RED ? RING : RED;
  static_assert(R >= 1 && J >= 1, "a CU has 160 KB of LDS");
};

// blockIdx.x: eight columns' upper halves, their lower halves, the next eight columns' ..; blockIdx.y: the slice of K
template <int MB, int MODE, int NT>
__global__ __launch_bounds__((QueueRowsCfg<MB, NT>::KL * 64)) void linear_queue_rows_kernel(
    const half_t* __restrict__ x, const void* __restrict__ Wp, float* __restrict__ part, int M, int N, int K,
    int tiles_per_wg, int stages_per_split, Epilogue epi) {
  using C = QueueRowsCfg<MB, NT>;
  constexpr int R = C::R, L = C::LOADS, KL = C::KL;
  extern __shared__ __attribute__((aligned(16))) char lds_queue[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = (blockIdx.x >> 3) & 1, col = (blockIdx.x >> 4) * 8 + (blockIdx.x & 7);
  const int ntiles = N >> 4, nst = K >> 6;
  const int tile_begin = col * tiles_per_wg;
  if (tile_begin >= ntiles) return;
  const int tile_end = min(ntiles, tile_begin + tiles_per_wg);
  const int m0 = half * (MB * 16);
  const int s_begin = blockIdx.y * stages_per_split, s_end = min(nst, s_begin + stages_per_split);
  const int n = s_begin + wave < s_end ? (s_end - s_begin - wave + KL - 1) / KL : 0;
  const char* wb[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
    wb[j] = (const char*)Wp + (int64_t)min(tile_begin + j, tile_end - 1) * nst * 2048 - (j % 2) * 2048;
  // (activations: load i takes rows 8 i .. 8 i + 7)
  uint32_t xo[2 * MB];
#pragma unroll
  for (int i = 0; i < 2 * MB; ++i) {
    const int row = min(m0 + i * 8 + (lane >> 3), M - 1);
    xo[i] = (uint32_t)row * (uint32_t)K * 2u + (uint32_t)(((lane & 7) ^ (4 * (i & 1) + (lane >> 4))) * 16);
  }
  const char* xb[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) xb[q] = (const char*)x - q * 1024;
  const char* ring = lds_queue + wave * (R * C::SLOT);
  const uint32_t ring_at = (uint32_t)(uintptr_t)(tq_lds_void*)lds_queue + wave * (R * C::SLOT);
  auto request = [&](int slot, int i) {
    const uint32_t st = (uint32_t)(s_begin + wave + KL * i);
    const uint32_t at = ring_at + slot * C::SLOT;
    const uint32_t wv = (uint32_t)lane * 16u + st * 2048u;
    tq_static_for<2 * NT>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      queue_load<(j % 4) * 1024, false>(wv, wb[j / 2], at + (j / 4) * 4096);
    });
    tq_static_for<2 * MB>([&](auto ic) {
      constexpr int f = decltype(ic)::value;
      queue_load<(f % 4) * 1024, false>(xo[f] + st * 128u, xb[f % 4], at + 2 * NT * 1024 + (f / 4) * 4096);
    });
  };
  float4_t acc[NT][MB];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[j][mb] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int r = 0; r < R; ++r)
    if (r < n) request(r, r);
  const int lr = lane & 15, lg = lane >> 4;
  const uint32_t x0 = lr * 128 + ((lg ^ (lr >> 1)) * 16), x1 = lr * 128 + (((4 + lg) ^ (lr >> 1)) * 16);
  int slot = 0;
  for (int i = 0; i < n; ++i) {
    if (i + R - 1 < n)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((R - 1) * L) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const char* from = ring + slot * C::SLOT;
    half8_t w[2][NT], xf[2][MB];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int j = 0; j < NT; ++j) w[u][j] = *reinterpret_cast<const half8_t*>(from + (2 * j + u) * 1024 + lane * 16);
#pragma unroll
      for (int f = 0; f < MB; ++f) xf[u][f] = *reinterpret_cast<const half8_t*>(from + (2 * NT + 2 * f) * 1024 + (u ? x1 : x0));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (i + R < n) request(slot, i + R);
    slot = slot == R - 1 ? 0 : slot + 1;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[j][mb] = mfma_16x16x32<MODE>(w[u][j], xf[u][mb], acc[j][mb]);
  }

  float4_t* red = reinterpret_cast<float4_t*>(lds_queue);
  constexpr int TOT = C::J * MB, PER = (TOT + KL - 1) / KL;
  constexpr bool AHEAD = PER <= (KL == 4 ? 10 : 4) && (!is_bf<MODE> || MODE == MODE_BF_POST);
#pragma unroll
  for (int j0 = 0; j0 < NT; j0 += C::J) {
    Ahead<MODE> ahead[AHEAD ? PER : 1];
    if (AHEAD && !part) {
#pragma unroll
      for (int q = 0; q < (AHEAD ? PER : 0); ++q) {
        const int p = min(wave + q * KL, TOT - 1);
        const int t = min(tile_begin + j0 + p / MB, tile_end - 1);
        ahead[q] = epilogue_ahead<MODE>(epi, min(m0 + p % MB * 16 + lr, M - 1), t * 16 + lg * 4);
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = j0; j < j0 + C::J && j < NT; ++j)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) red[((wave * C::J + j - j0) * MB + mb) * 64 + lane] = acc[j][mb];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int p = wave + q * KL, j = j0 + p / MB, mb = p % MB, t = tile_begin + j;
      if (p >= TOT || j >= NT || t >= tile_end) continue;
      float4_t sum = red[p * 64 + lane];
#pragma unroll
      for (int k = 1; k < KL; ++k) sum += red[(k * TOT + p) * 64 + lane];
      const int m = m0 + mb * 16 + lr, c = t * 16 + lg * 4;
      if (m >= M) continue;
      if (part)
        *reinterpret_cast<float4_t*>(part + ((int64_t)blockIdx.y * M + m) * N + c) = sum;
      else
        epilogue4<MODE, AHEAD>(epi, m, c, sum, ahead[AHEAD ? q : 0]);
    }
  }
}

template <int MB, bool W8, int MODE, int NT>
void launch_queue_cfg(const void* xp, const void* W, const void* scales, float* part, int S, int M, int N, int K,
                      int tiles_per_wg, int gx, int ks_per_split, const Epilogue& epi, hipStream_t s) {
  using C = QueueCfg<MB, W8, NT>;
  static_assert(C::SUMS_FIT, "queue_takes");
  static std::atomic<uint64_t> lds_allowed{0};  // one mask per instantiation
  auto kernel = linear_queue_kernel<MB, W8, MODE, NT>;
  if (!allow_lds((const void*)kernel, C::LDS_BYTES, lds_allowed)) return;  // the caller's launch check reports the error
  hipLaunchKernelGGL(kernel, dim3(gx, S), dim3(C::KL * 64), C::LDS_BYTES, s, (const half_t*)xp, W, (const half_t*)scales,
                     part, M, N, K, tiles_per_wg, ks_per_split, packed_row_blocks(M), epi);
}
template <int MB, bool W8, int MODE, int NT = 1>
void launch_queue_mb(const void* xp, const void* W, const void* scales, float* part, int S, int M, int N, int K,
                     int tiles_per_wg, int gx, int ks_per_split, const Epilogue& epi, hipStream_t s) {
  if constexpr (MB * NT <= 64 && (MB > 2 || (NT >= 5 && (W8 || MB == 2))))
    if (tiles_per_wg == NT)
      return launch_queue_cfg<MB, W8, MODE, NT>(xp, W, scales, part, S, M, N, K, tiles_per_wg, gx, ks_per_split, epi, s);
  if constexpr (NT < QUEUE_TILES)
    launch_queue_mb<MB, W8, MODE, NT + 1>(xp, W, scales, part, S, M, N, K, tiles_per_wg, gx, ks_per_split, epi, s);
}
template <int MB, int MODE, int NT = 1>
void launch_queue_rows_mb(const void* x, const void* W, float* part, int S, int M, int N, int K, int tiles_per_wg,
                          const Epilogue& epi, hipStream_t s) {
  if constexpr (NT < QUEUE_ROWS_TILES)
    if (tiles_per_wg > NT)
      return launch_queue_rows_mb<MB, MODE, NT + 1>(x, W, part, S, M, N, K, tiles_per_wg, epi, s);
  using C = QueueRowsCfg<MB, NT>;
  static std::atomic<uint64_t> lds_allowed{0};
  auto kernel = linear_queue_rows_kernel<MB, MODE, NT>;
  if (!allow_lds((const void*)kernel, C::LDS_BYTES, lds_allowed)) return;  // the caller's launch check reports the error
  const int columns = (N / 16 + tiles_per_wg - 1) / tiles_per_wg, stages = (K / 64 + S - 1) / S;
  hipLaunchKernelGGL(kernel, dim3((columns + 7) / 8 * 16, S), dim3(C::KL * 64), C::LDS_BYTES, s, (const half_t*)x, W, part,
                     M, N, K, tiles_per_wg, stages, epi);
}
}  // namespace

template <bool W8, int MODE>
void launch_queue(const void* xp, const void* W, const void* scales, float* part, int S, int M, int N, int K,
                  int tiles_per_wg, const Epilogue& epi, hipStream_t s) {
  const int ntiles = N / 16, nks = K / 32, gx = (ntiles + tiles_per_wg - 1) / tiles_per_wg;
  int ks_per_split = (nks + S - 1) / S;
  if (W8) ks_per_split = (ks_per_split + 1) & ~1;  // int8 blocks cover two steps
#define Q_RUN(MB)               \
  case MB:                      \
    return launch_queue_mb<MB, W8, MODE>(xp, W, scales, part, S, M, N, K, tiles_per_wg, gx, ks_per_split, epi, s)
  switch (queue_rows(M)) {
    case 1:  // int8 only
      if constexpr (W8)
        launch_queue_mb<1, W8, MODE>(xp, W, scales, part, S, M, N, K, tiles_per_wg, gx, ks_per_split, epi, s);
      return;
    Q_RUN(2);
    Q_RUN(3);
    Q_RUN(4);
    Q_RUN(5);
    Q_RUN(6);
    Q_RUN(7);
    Q_RUN(8);
  }
#undef Q_RUN
}

template <int MODE>
void launch_queue_rows(const void* x, const void* W, float* part, int S, int M, int N, int K, int tiles_per_wg,
                       const Epilogue& epi, hipStream_t s) {
  switch (queue_rows_blocks(M)) {
    case 5: return launch_queue_rows_mb<5, MODE>(x, W, part, S, M, N, K, tiles_per_wg, epi, s);
    case 6: return launch_queue_rows_mb<6, MODE>(x, W, part, S, M, N, K, tiles_per_wg, epi, s);
    case 7: return launch_queue_rows_mb<7, MODE>(x, W, part, S, M, N, K, tiles_per_wg, epi, s);
    default: return launch_queue_rows_mb<8, MODE>(x, W, part, S, M, N, K, tiles_per_wg, epi, s);
  }
}
