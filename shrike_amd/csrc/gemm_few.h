// The loop of products with few tokens (gemm_few.hip, moe_few.hip).
#pragma once

#include <type_traits>

#include "gemm_bf16.h"

namespace shk {

// A wavefront asks for everything before it waits for anything: its k-tiles at once where they fit its registers.
// acc += the wavefront's k-tiles (wave, wave + waves, ...) of RB blocks of 16 weight rows by NB blocks of 16 tokens.  wrow[]: the lane's
// weight row at its piece of the first tile.  C > 0: a wavefront has at most C tiles, which are all asked for at once;
// C = 0: batches of B tiles, two in flight.  Addresses are clamped into the matrices and what lies beyond k is
// zeroed when it is used: no load stands under a condition.
// rows(arow): the lane's token of every block, at its first element.  A token's piece `col` (a multiple of 8) lies at col * col_step.
template <int C, int B, int RB, int NB, typename Rows, typename Between>
__device__ __forceinline__ void few_multiply(f32x4 (&acc)[RB][NB], const u32x4* const (&wrow)[RB], Rows rows, int col_step, int k,
                                             int ktiles, int wave, int waves, Between between) {
  const int kg = threadIdx.x % kWave / 16;
  const bf16* arow[NB];
  rows(arow);
  constexpr int kTiles = C > 0 ? C : B;
  struct Batch {
    u32x4 w[kTiles][RB], x[kTiles][NB];
    uint32_t keep[kTiles];
  };
  auto load = [&](Batch& b, int t) {
#pragma unroll
    for (int u = 0; u < kTiles; ++u) {
      const int tt = t + u * waves, col = tt * 32 + kg * 8;
#pragma unroll
      for (int r = 0; r < RB; ++r)
        b.w[u][r] = __builtin_nontemporal_load(wrow[r] + static_cast<size_t>(tt < ktiles ? tt : ktiles - 1) * kWave);
      const bool inside = col < k;
      b.keep[u] = inside ? ~0u : 0u;
#pragma unroll
      for (int c = 0; c < NB; ++c)
        b.x[u][c] = *reinterpret_cast<const u32x4*>(arow[c] + (inside ? static_cast<size_t>(col) * col_step : 0));
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto multiply = [&](const Batch& b) {
#pragma unroll
    for (int u = 0; u < kTiles; ++u)
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        const u32x4 v = b.x[u][c] & b.keep[u];
#pragma unroll
        for (int r = 0; r < RB; ++r)
          acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, b.w[u][r]), __builtin_bit_cast(bf16x8, v),
                                                              acc[r][c], 0, 0, 0);
      }
  };
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int c = 0; c < NB; ++c) acc[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  Batch ping;
  load(ping, wave);
  if constexpr (C > 0) {
    between();
    multiply(ping);
  } else {
    Batch pong;
    const int step = B * waves, batches = (ktiles + step - 1) / step;
    load(pong, wave + step);
    between();
    int b = 0;
    for (; b + 3 < batches; b += 2) {
      multiply(ping);
      load(ping, wave + (b + 2) * step);
      multiply(pong);
      load(pong, wave + (b + 3) * step);
    }
    multiply(ping);
    if (b + 2 < batches) {
      load(ping, wave + (b + 2) * step);
      multiply(pong);
      multiply(ping);
    } else {
      multiply(pong);
    }
  }
}

constexpr int kFewTiles = 10, kFewPairs = 7;  // k-tiles of a wavefront that are held at once: of one block of weight rows, of two

// Element (row, token) of the 16 x 16 results that `waves` wavefronts have left in LDS, added in their order.
__device__ __forceinline__ float few_sum(const f32x4* red, int stride, int row, int token, int waves) {
  const float* p = reinterpret_cast<const float*>(red + row / 4 * 16 + token) + row % 4;
  float v = 0.f;
#pragma unroll 4
  for (int w = 0; w < waves; ++w) v += p[static_cast<size_t>(w) * stride * 4];
  return v;
}

// Wavefronts that share k (or walks of it, where a wavefront takes two; the figures are with one each): where four to eight of them hold
// all their tiles at once, the number that holds the fewest beyond k, else four or five.  Few, because each more is another sum to add
// at the end: 896 x 896 with one token 2.97 us in 4, 3.10 in 7, 3.21 in 15; 3584 x 18944 at 1 / 8 / 16 tokens 22.2 / 23.2 / 27.0 in 4, 22.0 / 24.1 / 28.4 in 5, 23.1 / 24.5 / 27.8
// in 16; 1536 x 8960, whose 280 tiles five share without loads beyond k, 9.7 / 9.8 / 10.6 in 4 and 9.0 / 9.2 / 11.0 in 5.
// (Whatever the tokens: a row's bits do not depend on those beside it.)
inline int few_waves(int ktiles, int most) {
  int best = 0, least = 0;
  for (int waves = 4; waves <= 8; ++waves) {
    const int tiles = (ktiles + waves - 1) / waves;
    if (tiles <= most && (!best || tiles * waves < least)) best = waves, least = tiles * waves;
  }
  const auto whole = [&](int waves) { return (ktiles + 4 * waves - 1) / (4 * waves) * 4 * waves; };
  return best ? best : whole(5) <= whole(4) ? 5 : 4;
}

// fn with the number of k-tiles of a wavefront as a constant, 0 for more than MOST.
template <int MOST, int C = 1, typename Fn>
void with_tiles(int tiles, Fn fn) {
  if constexpr (C > MOST) {
    fn(std::integral_constant<int, 0>{});
  } else {
    if (tiles == C) fn(std::integral_constant<int, C>{});
    else with_tiles<MOST, C + 1>(tiles, fn);
  }
}

}  // namespace shk
