// bfloat16 products of more than 64 tokens, with weights in the tiled layout that gemm_bf16.hip describes: wide_loop()
// of gemm_wide.h in eight tile sizes.
//
// The results leave through LDS in whole 16-byte pieces along the rows, by straight-line code without a branch per
// value: 2 to 5 us a workgroup, 20 to 30 where every value was tested and stored for itself.  Other epilogues and rows that are no
// whole pieces finish eight rows at a time: 4864 x 896 at 1,119 tokens with bounded gates 33 us in the kernel before, 46 one value at a
// time, 29 so; 4737 x 896 at 2,048 47, 63, 36; added to 9472 x 3584 float32 results at 2,048 199, 256, 142.
// Gates other than SiLU, or with constants, leave from registers too: 9472 x 3584 at 1,501 tokens in two launches 102.7 and 82.3 us behind
// that loop, 99.1 and 78.0 so.
// Against the kernel before (16 wavefronts, tiles of 16 x 16, 256 x 256, 256 x 128 and 128 x 128), both in the passes of whole models on
// one card: 7B at 2,048 tokens QKV 100 us -> 67, output and down 168 -> 146 on average, gate/up 507 -> 462 (1.20 PFLOP/s); at 512
// QKV 46 -> 26, output 33 -> 25, gate/up 156 -> 133 (two launches), down 104 -> 78; 14B at 512 QKV 64 -> 58, output and down
// 72 -> 58, gate/up 156 -> 126.  Alone, replayed on the same operands, a product takes 2 to 10 % less.
#include "gemm_bf16.h"
#include "gemm_wide.h"

#include <algorithm>
#include <type_traits>

namespace shk {

// WHOLE: rows in whole 16-byte pieces, finished in registers: at most a bias or SiLU's gate, or (kWholeGates) bfloat16 rows of any gate,
// its constants in `bias`.  Anything else is a kernel of its own, which keeps all short.  pieces: its results leave in 16-byte pieces too.
constexpr int kWholeGates = 2;
template <int GM, int GN, int RM, int RN, bool GATED, int WHOLE>
__global__ void __launch_bounds__(GM* GN* kWave) __attribute__((amdgpu_waves_per_eu(GM * GN / 4, GM * GN / 4)))
    gemm_wide_kernel(const bf16* __restrict__ a, int lda, int n, int k, const uint4* __restrict__ wt, int ktiles, int m,
                     const float* __restrict__ bias, void* __restrict__ out, int ldo, int out_f32, int accumulate, int pieces,
                     TileOrder order) {
  using S = WideShape<GM, GN, RM, RN>;
  constexpr int WL = S::kWLoads, XL = S::kXLoads;
  __shared__ u32x4 mem[S::kLds / 16];
  const int tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wm = wave / GN, wn = wave % GN;
  int tile_x, tile_y, share;
  if (!big_tile(order, tile_x, tile_y, share)) return;
  const int ksplit = order.shares;
  const int mb0 = tile_x * S::kTiles, tok0 = tile_y * (32 * GN * RN);
  // blocks of 16 weight rows; a gated weight has two per 16 output rows
  const int mblocks = (GATED ? 2 : 1) * ((m + 15) / 16);
  // this share's stages of k; the last stage of k may be half a one
  const int all = (ktiles + 1) / 2;
  const int first = static_cast<int>(static_cast<long long>(all) * share / ksplit);
  const int stages = static_cast<int>(static_cast<long long>(all) * (share + 1) / ksplit) - first;
  if (stages == 0) {  // more shares than stages: zeros
    float* o = static_cast<float*>(out) + static_cast<size_t>(share) * n * ldo;
    for (int i = tid; i < 32 * GN * RN * 16 * S::kTiles; i += S::kWaves * kWave) {
      const int token = tok0 + i / (16 * S::kTiles), row = mb0 * 16 + i % (16 * S::kTiles);
      if (token < n && row < m) o[static_cast<size_t>(token) * ldo + row] = 0.f;
    }
    return;
  }
  const int left = ktiles - 2 * first, subs = 2 * stages < left ? 2 * stages : left;

  // What a wavefront loads: weight tiles and units of 8 tokens wave, wave + kWaves, ..., from rows clamped into the
  // matrices (their products are never stored).  In the last stage of k a piece beyond k is replaced by the
  // stage's first (numbers that meet the zeros which pad the weight tiles).
  unsigned woff[WL], xoff[2 * XL];
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int rb = wave + S::kWaves * i;
    const int block = mb0 + rb < mblocks ? rb : mblocks - 1 - mb0;
    woff[i] = (static_cast<unsigned>(block) * ktiles * kWave + lane) * 16u;
  }
  const unsigned piece = (lane % 8) ^ (lane / 8);
#pragma unroll
  for (int i = 0; i < 2 * XL; ++i) {
    const int t = (wave + S::kWaves * i) * 8 + lane / 8;
    const int token = tok0 + t < n ? t : n - 1 - tok0;
    xoff[i] = static_cast<unsigned>(token) * lda * 2u + piece * 16u;
  }
  const unsigned beyond = (all - 1) * 64 + static_cast<int>(piece) * 8 < k ? 0u : piece * 16u;
  const char* wsrc = reinterpret_cast<const char*>(wt) + (static_cast<size_t>(mb0) * ktiles + 2 * first) * 1024;
  const char* xsrc = reinterpret_cast<const char*>(a) + static_cast<size_t>(tok0) * lda * 2 + static_cast<size_t>(first) * 128;

  f32x16 acc[RM][RN];
  wide_loop<GM, GN, RM, RN>(acc, mem, wsrc, woff, xsrc, xoff, beyond, all - 1 - first, subs, stages);

  // Accumulator register g * 4 + r of lane (j, half): token j, row g * 8 + half * 4 + r.  Gated: rows 0 to 15 of a tile
  // belong to the gate, 16 to 31 are the same rows of the other factor.
  constexpr int kRows = (GATED ? 16 : 32) * RM;  // output rows of a wavefront
  const int half = lane / 32, j = lane % 32;
  const int row0 = (GATED ? mb0 / 2 : mb0) * 16 + wm * kRows, tok = tok0 + wn * RN * 32;
  const size_t plane = static_cast<size_t>(share) * n;
  if (row0 >= m) return;  // (no barrier follows)
  char* mine = reinterpret_cast<char*>(&mem[0]) + wave * (32 * (32 * RM * 4 + 16));
  if constexpr (WHOLE) {
    const float limit = WHOLE == kWholeGates && bias ? bias[0] : 0.f, shift = WHOLE == kWholeGates && bias ? bias[1] : 0.f;
    auto gated = [&](float g, float u, auto act) {
      if constexpr (WHOLE == kWholeGates) {
        g = limit > 0.f ? fminf(g, limit) : g, u = limit > 0.f ? fminf(fmaxf(u, -limit), limit) : u;
        u = bias ? u + shift : u;
      }
      return gate_times_up(g, u, decltype(act)::value, nullptr);
    };
    auto finish = [&](auto f32, auto biased, auto act) {
      constexpr bool F32 = decltype(f32)::value, BIASED = decltype(biased)::value;
      // (asked for together: one by one, each group of rows waits for its own)
      f32x4 add[RM][4];
      if constexpr (BIASED) {
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const int row = row0 + 32 * i + g * 8 + half * 4;
            add[i][g] = *reinterpret_cast<const f32x4*>(bias + (row < m ? row : m - 4));
          }
      }
      constexpr int E = F32 ? 4 : 2, kPitch = kRows * E + 16, kPieces = kRows * E / 16;
      auto put = [&](const f32x16 (&c)[RN], int jn, int i) {
#pragma unroll
        for (int g = 0; g < (GATED ? 2 : 4); ++g) {
          const int row = (GATED ? 16 : 32) * i + g * 8 + half * 4;
          f32x4 v;
#pragma unroll
          for (int r = 0; r < 4; ++r)
            v[r] = GATED ? gated(c[jn][g * 4 + r], c[jn][(GATED ? 8 : 0) + g * 4 + r], act) : c[jn][g * 4 + r];
          if constexpr (BIASED) v += add[i][g];
          if constexpr (F32) {
            *reinterpret_cast<f32x4*>(mine + j * kPitch + row * 4) = v;
          } else {
            bf16x4 o;
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] = static_cast<__bf16>(v[r]);
            *reinterpret_cast<bf16x4*>(mine + j * kPitch + row * 2) = o;
          }
        }
      };
#pragma unroll
      for (int jn = 0; jn < RN; ++jn) {
        put(acc[0], jn, 0);
        put(acc[1], jn, 1);
        if constexpr (RM > 2) put(acc[2], jn, 2);
        if constexpr (RM > 3) put(acc[3], jn, 3);
        SHK_LDS_DONE();
#pragma unroll
        for (int q = 0; q < 32 * kPieces / kWave; ++q) {
          const int at = q * kWave + lane, t = at / kPieces, p = at % kPieces, token = tok + jn * 32 + t, row = row0 + p * (16 / E);
          const u32x4 v = *reinterpret_cast<const u32x4*>(mine + t * kPitch + p * 16);
          if (token < n && row < m)
            *reinterpret_cast<u32x4*>(static_cast<char*>(out) + ((plane + token) * ldo + row) * E) = v;
        }
        SHK_LDS_DONE();
      }
    };
    constexpr std::integral_constant<int, kActSilu> silu;
    auto leave = [&](auto f32) {
      if (!GATED && bias)
        finish(f32, std::bool_constant<!GATED>{}, silu);
      else
        finish(f32, std::false_type{}, silu);
    };
    if constexpr (WHOLE == kWholeGates) {
      const std::false_type no;
      if (accumulate == kActQuickGelu)
        finish(no, no, std::integral_constant<int, kActQuickGelu>{});
      else if (accumulate == kActGeluTanh)
        finish(no, no, std::integral_constant<int, kActGeluTanh>{});
      else if (accumulate == kActRelu)
        finish(no, no, std::integral_constant<int, kActRelu>{});
      else
        finish(no, no, silu);
    } else if (out_f32) {
      leave(std::true_type{});
    } else {
      leave(std::false_type{});
    }
    return;
  }
  // Anything else: the sums go through LDS as they are; a lane finishes eight neighbouring rows of a token at a time, so that
  // what is the same for all of them is asked once, and stores them as 16-byte pieces where rows allow.  Others go
  // back to their place and leave as single values, neighbouring lanes on neighbouring rows.
  constexpr int kPitch = 32 * RM * 4 + 16;
  auto place = [&](int t, int p) { return reinterpret_cast<float*>(mine + t * kPitch) + (GATED ? p / 16 * 32 + p % 16 : p); };
  auto put = [&](const f32x16 (&c)[RN], int jn, int i) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4 v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = c[jn][g * 4 + r];
      *reinterpret_cast<f32x4*>(mine + j * kPitch + (i * 32 + g * 8 + half * 4) * 4) = v;
    }
  };
  const int done = pieces ? m & ~7 : 0;  // rows below it leave in pieces
  const float limit = GATED && bias ? bias[0] : 0.f, shift = GATED && bias ? bias[1] : 0.f;
  const bool near_bias = reinterpret_cast<uintptr_t>(bias) % 16 == 0;
  auto finish = [&](float (&v)[8], const float (&u)[8], int row) {
    if constexpr (GATED) {
      float g[8], f[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        g[e] = v[e], f[e] = u[e];
        if (limit > 0.f) g[e] = fminf(g[e], limit), f[e] = fminf(fmaxf(f[e], -limit), limit);
        if (bias) f[e] += shift;
      }
      auto all = [&](auto act) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = gate_times_up(g[e], f[e], decltype(act)::value, nullptr);
      };
      if (accumulate == kActSilu)
        all(std::integral_constant<int, kActSilu>{});
      else if (accumulate == kActGeluTanh)
        all(std::integral_constant<int, kActGeluTanh>{});
      else if (accumulate == kActRelu)
        all(std::integral_constant<int, kActRelu>{});
      else
        all(std::integral_constant<int, kActQuickGelu>{});
    } else {
      if (bias && row + 8 <= m && near_bias) {
        const f32x4 lo = *reinterpret_cast<const f32x4*>(bias + row), hi = *reinterpret_cast<const f32x4*>(bias + row + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += lo[e], v[4 + e] += hi[e];
      } else if (bias) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += bias[row + e < m ? row + e : m - 1];
      }
      if (accumulate == kPlainReluSquared) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = plain_act(v[e], kPlainReluSquared, row + e);
      } else if (accumulate >= kPlainSiluRows && row < accumulate / kPlainSiluRows) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = plain_act(v[e], accumulate, row + e);
      }
    }
  };
#pragma unroll
  for (int jn = 0; jn < RN; ++jn) {
    put(acc[0], jn, 0);
    put(acc[1], jn, 1);
    if constexpr (RM > 2) put(acc[2], jn, 2);
    if constexpr (RM > 3) put(acc[3], jn, 3);
    SHK_LDS_DONE();
#pragma unroll 1
    for (int at = lane; at < 4 * kRows; at += kWave) {
      const int t = at / (kRows / 8), p = at % (kRows / 8) * 8, token = tok + jn * 32 + t, row = row0 + p;
      if (token >= n || row >= m) continue;
      f32x4* from = reinterpret_cast<f32x4*>(place(t, p));
      const f32x4 lo = from[0], hi = from[1];
      float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}, u[8] = {};
      if constexpr (GATED) {
        const f32x4 ulo = from[4], uhi = from[5];
#pragma unroll
        for (int e = 0; e < 4; ++e) u[e] = ulo[e], u[4 + e] = uhi[e];
      }
      finish(v, u, row);
      const size_t idx = (plane + token) * ldo + row;
      if (row >= done) {
        from[0] = f32x4{v[0], v[1], v[2], v[3]}, from[1] = f32x4{v[4], v[5], v[6], v[7]};
      } else if (out_f32) {
        f32x4* o = reinterpret_cast<f32x4*>(static_cast<float*>(out) + idx);
        f32x4 x = {v[0], v[1], v[2], v[3]}, y = {v[4], v[5], v[6], v[7]};
        if (accumulate == 1 && !GATED) x = o[0] + x, y = o[1] + y;
        o[0] = x, o[1] = y;
      } else {
        bf16x8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = static_cast<__bf16>(v[e]);
        *reinterpret_cast<bf16x8*>(static_cast<bf16*>(out) + idx) = o;
      }
    }
    SHK_LDS_DONE();
    const int tokens = n - (tok + jn * 32) < 32 ? n - (tok + jn * 32) : 32;
    if (row0 + kRows > done && done < m) {
#pragma unroll
      for (int q = 0; q < (kRows + kWave - 1) / kWave; ++q) {
        const int p = q * kWave + lane, row = row0 + p;
        if (p >= kRows || row < done || row >= m) continue;
        const float* from = place(0, p);
        const size_t idx = (plane + tok + jn * 32) * ldo + row;
        auto leave = [&](auto* o, auto added) {
#pragma unroll 8
          for (int t = 0; t < tokens; ++t, o += ldo, from += kPitch / 4) {
            if constexpr (decltype(added)::value)
              *o = *o + *from;
            else
              *o = from_float<std::remove_pointer_t<decltype(o)>>(*from);
          }
        };
        if (!out_f32)
          leave(static_cast<bf16*>(out) + idx, std::false_type{});
        else if (accumulate == 1 && !GATED)
          leave(static_cast<float*>(out) + idx, std::true_type{});
        else
          leave(static_cast<float*>(out) + idx, std::false_type{});
      }
    }
    SHK_LDS_DONE();
  }
}

// A price of few shares of a long k: the least time, at 7 TB/s, of the dies' fetches in an order in which tiles are no longer dealt out (every eighth
// tile a die's, rectangles where the numbers divide).  In the present order (tile_of) fetches bound none of these sizes, and whether numbers
// divide changes nothing but this price.  It stays because the choices that it makes are not the worse ones: with the shares that it gives and with those that
// wide_time() gives alone, product without its reader, 896 x 18944 at 2,048 tokens 4 shares 64.6 us and 3 69.3, at 2,112 5 71.3 and 3 73.7, at 2,752 4
// 90.4 and 2 93.4, 640 x 18944 at 2,048 6 47.8 and 4 52.3, 1152 x 18944 3 83.6 and 2 96.5, 896 x 9472 4 36.3 and 3 36.6; against it 896 x 18944 at 3,712, two shares
// in tiles of 256 x 128 123.9 and 128 x 256 112.9, and 2304 x 9472 at 777 2 46.8 and 4 38.6.  The jumps at 3584 x 18944 (one share at 1,700, two at 1,792, one at
// 1,793: 216, 210, 225 us, 210, 221, 214 with the other number) are wide_time()'s own.  With less than 8,192 of k the shares' start and end weigh more
// (896 x 4864 at 1,119 tokens in a prompt, in the old order: 25 us in the three shares of 128 x 128 without this, 31 in the two of 128 x 192 that it would take;
// 19 now).
static double wide_fetch(const WideTile& t, int n, int wblocks, int k) {
  const int tiles_x = (wblocks * 16 + t.rows - 1) / t.rows, tiles_y = (n + t.tokens - 1) / t.tokens;
  if (tiles_y <= 2 || k < 8192) return 0.0;
  return 2.0 + t.ends + ((k + 63) / 64) * 128.0 * big_operands(tiles_x, tiles_y, t.rows, t.tokens) / 7e6;
}

static double wide_estimate(const WideTile& t, int split, int n, int wblocks, int k) {
  const long long groups = static_cast<long long>((wblocks * 16 + t.rows - 1) / t.rows) * ((n + t.tokens - 1) / t.tokens) * split;
  const double us = wide_time(t, static_cast<double>(groups), ((k + 63) / 64 + split - 1) / split);
  return split > 1 ? std::max(us, wide_fetch(t, n, wblocks, k)) : us;
}

// The tile of the least estimate.
static int wide_tile(int split, int n, int wblocks, int k, double* least) {
  int best = 0;
  *least = wide_estimate(kWide[0], split, n, wblocks, k);
  for (int i = 1; i < kWideTiles; ++i) {
    const double us = wide_estimate(kWide[i], split, n, wblocks, k);
    if (us < *least) *least = us, best = i;
  }
  return best;
}

// Tiles that do not make whole rounds of the compute units (256 x 256 tiles of the 7B gate/up matrix at 512 tokens: 296) are
// better run as two products: the rows whose tiles make whole rounds, then the others with the tile that suits them.
struct WidePlan {
  int tile, main_blocks, rest_tile;  // main_blocks: blocks of 16 weight rows of the first product, 0: one product
};
static WidePlan wide_plan(int split, int n, int wblocks, int k, double* us) {
  n = counted_tokens(n);
  WidePlan plan = {0, 0, 0};
  plan.tile = wide_tile(split, n, wblocks, k, us);
  if (split > 1) return plan;
  const double whole = *us;
  for (int i = 0; i < kWideTiles; ++i) {
    const WideTile& t = kWide[i];
    const int tiles_x = (wblocks * 16 + t.rows - 1) / t.rows, tiles_y = (n + t.tokens - 1) / t.tokens;
    const long long total = static_cast<long long>(tiles_x) * tiles_y;
    const int main_x = static_cast<int>(total / t.units * t.units / tiles_y);
    if (total <= t.units || main_x <= 0 || main_x >= tiles_x) continue;
    const int main_blocks = main_x * (t.rows / 16);
    double rest;
    const int rest_tile = wide_tile(1, n, wblocks - main_blocks, k, &rest);
    const double both = wide_estimate(t, 1, n, main_blocks, k) + rest;
    if (both < 0.97 * whole && both < *us) *us = both, plan = {i, main_blocks, rest_tile};
  }
  return plan;
}

// Shares of k: at most 16, of at least 16 tiles of 32, that the estimate expects to be the fastest with what writing and
// reading the output costs: float32 parts, or `whole_bytes` a value of an unsplit product (3 TB/s).
int wide_splits(int n, int m, int k, int whole_bytes) {
  const int mblocks = (m + 15) / 16, ktiles = (k + 31) / 32;
  const int most = ktiles / 16 < 16 ? ktiles / 16 : 16;
  int best = 1;
  double least;
  const WidePlan whole = wide_plan(1, n, mblocks, k, &least);
  if (!whole.main_blocks) least = std::max(least, wide_fetch(kWide[whole.tile], counted_tokens(n), mblocks, k));
  const double values = static_cast<double>(counted_tokens(n)) * m;
  least += 2.0 * values * whole_bytes / 3e6;
  for (int split = 2; split <= most; ++split) {
    double us;
    wide_plan(split, n, mblocks, k, &us);
    us += 2.0 * values * split * 4.0 / 3e6;
    if (us < 0.97 * least) least = us, best = split;  // more shares only for a clear gain
  }
  return best;
}

int wide_parts(int n, int m, int k, int gated) {
  double us;
  return wide_plan(1, n, (gated ? 2 : 1) * ((m + 15) / 16), k, &us).main_blocks ? 2 : 1;
}

// The tile of a product's only or first launch, and 16 * (1 + the tile of its second, where there is one).
int wide_tiles(int n, int m, int k, int gated, int ksplit) {
  double us;
  const WidePlan plan = wide_plan(ksplit, n, (gated ? 2 : 1) * ((m + 15) / 16), k, &us);
  return plan.tile + (plan.main_blocks ? 16 * (1 + plan.rest_tile) : 0);
}

void wide_tile_size(int tile, int* rows, int* tokens) { *rows = kWide[tile].rows, *tokens = kWide[tile].tokens; }

// Whether offsets within a tile fit 32 bits.
bool wide_serves(int lda, int k) { return lda <= 4 * 1024 * 1024 && k <= 4 * 1024 * 1024; }

template <int GM, int GN, int RM, int RN>
static void launch_wide(hipStream_t s, const bf16* a, int lda, int n, int k, const uint4* wt, int m, int wblocks, const float* bias,
                        void* out, int ldo, int out_f32, int accumulate, int gated, int ksplit) {
  using S = WideShape<GM, GN, RM, RN>;
  const int tiles_x = (wblocks + S::kTiles - 1) / S::kTiles, tiles_y = (n + 32 * GN * RN - 1) / (32 * GN * RN);
  TileOrder order;
  const unsigned groups = big_grid(tiles_x, tiles_y, ksplit, 16 * S::kTiles, 32 * GN * RN, k, S::kLds <= 80 * 1024 ? 512 : 256, &order);
  const int per = out_f32 ? 4 : 8;  // values of 16 bytes
  const int pieces = ldo % per == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
  const bool rows = pieces && m % per == 0;
  const bool whole = rows && reinterpret_cast<uintptr_t>(bias) % 16 == 0 && (gated ? accumulate == kActSilu && !bias : accumulate == 0);
  const int ktiles = (k + 31) / 32;
  const auto kernel = gated ? (whole                ? gemm_wide_kernel<GM, GN, RM, RN, true, 1>
                               : rows && !out_f32 ? gemm_wide_kernel<GM, GN, RM, RN, true, kWholeGates>
                                                  : gemm_wide_kernel<GM, GN, RM, RN, true, 0>)
                            : (whole ? gemm_wide_kernel<GM, GN, RM, RN, false, 1> : gemm_wide_kernel<GM, GN, RM, RN, false, 0>);
  kernel<<<groups, S::kWaves * kWave, 0, s>>>(a, lda, n, k, wt, ktiles, m, bias, out, ldo, out_f32, accumulate, pieces,
                                                            order);
}

void wide_product(hipStream_t s, const bf16* a, int lda, int n, int k, const uint4* wt, int m, const float* bias, void* out,
                  int ldo, int out_f32, int accumulate, int gated, int ksplit) {
  static decltype(&launch_wide<2, 2, 2, 2>) const launch[kWideTiles] = {
      launch_wide<2, 4, 4, 2>, launch_wide<2, 2, 4, 3>, launch_wide<2, 2, 3, 4>, launch_wide<2, 2, 3, 3>,
      launch_wide<4, 2, 2, 2>, launch_wide<2, 2, 2, 4>, launch_wide<2, 2, 2, 3>, launch_wide<2, 2, 2, 2>};
  const int wblocks = (gated ? 2 : 1) * ((m + 15) / 16);
  double us;
  const WidePlan plan = wide_plan(ksplit, n, wblocks, k, &us);
  if (!plan.main_blocks) {
    launch[plan.tile](s, a, lda, n, k, wt, m, wblocks, bias, out, ldo, out_f32, accumulate, gated, ksplit);
    return;
  }
  const int main_rows = plan.main_blocks * 16 / (gated ? 2 : 1);
  launch[plan.tile](s, a, lda, n, k, wt, main_rows, plan.main_blocks, bias, out, ldo, out_f32, accumulate, gated, 1);
  // (a gated product's `bias` is its gate's two constants, the same for every row)
  launch[plan.rest_tile](s, a, lda, n, k, wt + static_cast<size_t>(plan.main_blocks) * ((k + 31) / 32) * kWave, m - main_rows,
                            wblocks - plan.main_blocks, bias && !gated ? bias + main_rows : bias,
                            static_cast<char*>(out) + static_cast<size_t>(main_rows) * (out_f32 ? 4 : 2), ldo, out_f32,
                            gated ? accumulate : plain_act_from(accumulate, main_rows), gated, 1);
}

}  // namespace shk
