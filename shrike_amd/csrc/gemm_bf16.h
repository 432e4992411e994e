// What the kernels of bfloat16 products share: operand types, activations in their epilogues, and the order in which
// the large ones take their tiles.
#pragma once

#include "api.h"
#include "common.h"

namespace shk {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
// 16 bytes as the compiler's own vector type: copies of it are loads and stores,
// where copies of HIP's uint4 struct can end up as memcpy through scratch memory
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float silu(float g) { return g / (1.f + __expf(-g)); }

// The activation of a gated product's gate: kActSilu, or the tanh form of GELU,
// 0.5 g (1 + tanh(sqrt(2/pi) (g + 0.044715 g^3))) = g / (1 + exp(-2 u)).  Gated
// kernels get the code in the argument that other products use for `accumulate`
// (a gated product never accumulates).
// kActRelu is max(g, 0), kActQuickGelu g / (1 + exp(-1.702 g)).
constexpr int kActSilu = 1, kActGeluTanh = 2, kActRelu = 3, kActQuickGelu = 4;
__device__ __forceinline__ float gate_act(float g, int act) {
  if (act == kActGeluTanh) {
    const float u = 0.7978845608028654f * (g + 0.044715f * g * g * g);
    return g / (1.f + __expf(-2.f * u));
  }
  if (act == kActRelu) return fmaxf(g, 0.f);
  if (act == kActQuickGelu) return g / (1.f + __expf(-1.702f * g));
  return silu(g);
}

// The activation of a plain product: such a product's `accumulate` argument is 0 (store), 1 (add to a
// float32 output), kPlainReluSquared: the square of max(v, 0) is stored, v the sum with its bias, or 4 *
// rows: the first `rows` output rows (weight rows) pass SiLU, the others are stored as they are.
constexpr int kPlainReluSquared = 2, kPlainSiluRows = 4;
__device__ __forceinline__ float plain_act(float v, int accumulate, int row) {
  if (accumulate == kPlainReluSquared) {
    const float r = fmaxf(v, 0.f);
    return r * r;
  }
  return accumulate >= kPlainSiluRows && row < accumulate / kPlainSiluRows ? silu(v) : v;
}
// act(g) * u of a gated product.  A gate with constants brings them where other products bring their bias
// (a gated product has none): args[0] > 0 bounds the gate from above and the other factor from both sides
// before anything else, args[1] is added to that factor.
__device__ __forceinline__ float gate_times_up(float g, float u, int act, const float* __restrict__ args) {
  if (args) {
    const float limit = args[0];
    if (limit > 0.f) {
      g = fminf(g, limit);
      u = fminf(fmaxf(u, -limit), limit);
    }
    u += args[1];
  }
  return gate_act(g, act) * u;
}

constexpr int kDies = 8;        // accelerator dies (XCDs), each with an L2 of its own
constexpr int kDieUnits = 32;  // compute units per die

// i / by for i < 2^31 and a number `by` that the host knows: the upper half of a product, exact since times exceeds 2^(31 + shift) / by by less
// than one and 2^shift is at least `by`.  (A division by a number known at run time only is a chain of some 25 instructions.)
struct Divisor {
  unsigned times, shift;
};
inline Divisor divisor(unsigned by) {
  unsigned shift = 0;
  while (1ull << shift < by) ++shift;
  return Divisor{static_cast<unsigned>(((1ull << (31 + shift)) + by - 1) / by), shift};
}
__host__ __device__ __forceinline__ int divided(int i, const Divisor& d) {
  return static_cast<int>(static_cast<unsigned>(static_cast<unsigned long long>(2u * static_cast<unsigned>(i)) * d.times >> 32) >> d.shift);
}

// How the tiles of a large product (tiles_x along the weight rows, tiles_y along the tokens, `shares` of k) are dealt out: in one row,
// share by share (or, with one row of token tiles, tile by tile), within a share in `strips` runs of neighbouring token tiles, the taller ones first, within a
// strip weight tile by weight tile.  in_turn: dies take 32 of them at a time, in turn, else an eighth of the row each.
struct TileOrder {
  int tiles_x, tiles_y, shares, strips, in_turn;
  // Tiles of all shares and of one; token tiles (with one row of them: shares) of a low strip, of all taller ones, and those ones' tiles.
  int all, each, low, tall_rows, tall_tiles;
  Divisor by_each, by_strip[2], by_high[2];  // (of low strips and of taller ones)
};

// The tile of workgroup `group` of the large kernels; false: none (the grid is padded).
// Workgroups are handed to the chip's eight dies (each with its own L2) in turn, workgroup p to die p % 8.  Die d takes the d-th
// eighth of the row of tiles, in order: what its 32 compute units work on at a time is a run of neighbours that share operands, so that
// its L2 serves most of their loads, whatever the numbers of tiles.  All dies together draw 10 TB/s from beyond their L2s, 40 GB/s a
// compute unit, which takes in 130 to 150 from its L2.  Against rectangles for the dies where the numbers divided, and every eighth tile on a
// die where not, weights cold: 896 x 4864 at 700 / 1,119 / 2,048 tokens 19.0 / 25.1 / 34.3 us -> 15.1 / 19.2 / 28.6, 3584 x 18944 at 512
// 76.3 -> 73.2, gate and up of 18944 x 3584 at 300 117 -> 102; whole prompts of the 7B sizes at 2,048 tokens 26.6 -> 26.1 ms.
// Nothing of a workgroup can begin before this is known, so it holds no divisions and nothing to branch on but the padding: 896 x 896 at 777 / 1,119 /
// 2,048 tokens 8.8 / 8.8 / 9.0 us with both, 8.5 / 8.5 / 8.7 so, 4096 10.4 and 9.9; 1152 x 896 at 512 8.7 and 8.4; 896 x 4864 at 1,119 16.3 and 15.9.
// One row of token tiles: no two tiles of a share have weights in common, and a die that walks one share after the other asks for all of a moment's
// weights from the same part of every row of tiles.  So a tile's shares follow each other, as its token tiles would: 4096 x 4096 in four at 65 / 100 / 128
// tokens 15.6 / 16.5 / 17.1 us share by share, 14.8 / 15.5 / 16.0 so, 2048 x 4096 10.6 / 10.9 / 11.0 and 10.3 / 10.6 / 10.6.
__host__ __device__ __forceinline__ bool tile_of(const TileOrder& t, unsigned group, int& tile_x, int& tile_y, int& share) {
  const int die = group % kDies, turn = group / kDies;
  const int eighth = static_cast<unsigned>(t.all) / kDies, over = static_cast<unsigned>(t.all) % kDies;
  const int begin = eighth * die + over * die / kDies, end = eighth * (die + 1) + over * (die + 1) / kDies;
  int i = t.in_turn ? (turn / kDieUnits * kDies + die) * kDieUnits + turn % kDieUnits : begin + turn;
  if (i >= (t.in_turn ? t.all : end)) return false;
  share = divided(i, t.by_each);
  i -= share * t.each;
  const bool tall = i < t.tall_tiles;
  i -= tall ? 0 : t.tall_tiles;
  const int high = t.low + tall, strip = divided(i, tall ? t.by_strip[1] : t.by_strip[0]);
  i -= strip * high * t.tiles_x;
  tile_x = divided(i, tall ? t.by_high[1] : t.by_high[0]);
  tile_y = (tall ? 0 : t.tall_rows) + strip * high + i - tile_x * high;
  if (t.tiles_y == 1) share = tile_y, tile_y = 0;
  return true;
}

__device__ __forceinline__ bool big_tile(const TileOrder& t, int& tile_x, int& tile_y, int& share) {
  return tile_of(t, blockIdx.x, tile_x, tile_y, share);
}

// The grid of the large kernels, and the strips with which the tiles that a die works on at a time (`units`: workgroups on the whole
// chip) need the fewest rows of weights and activations.  In turn from four rounds of tiles on with up to 2,048 of k: all dies then work on one strip, and
// a die meets the same few weight tiles in every strip, which with so short a k stay in its L2.  An eighth each and in turn: 8192 x 1024 at 8,192 / 16,384
// tokens 131 / 268 us and 125 / 244, 16384 x 1024 at 4,096 / 16,384 130 / 525 and 124 / 486, 9728 x 896 at 16,384 281 and 262; with longer k, gate and up of
// 18944 x 3584 at 2,048 / 4,096 435 / 862 and 449 / 880.
inline unsigned big_grid(int tiles_x, int tiles_y, int shares, int tile_rows, int tile_tokens, int k, int units, TileOrder* order) {
  const long long all = static_cast<long long>(tiles_x) * tiles_y * shares, each = (all + kDies - 1) / kDies;
  const int in_turn = static_cast<long long>(tiles_x) * tiles_y >= 4 * kDies * kDieUnits && k <= 2048;
  const int most = in_turn ? kDieUnits : units / kDies, at_once = static_cast<int>(each < most ? each : most);
  int best = 1;
  long long least = 0;
  for (int strips = 1; strips <= tiles_y; ++strips) {
    const int high = (tiles_y + strips - 1) / strips, wide = (at_once + high - 1) / high;
    const long long rows = static_cast<long long>(wide < tiles_x ? wide : tiles_x) * tile_rows +
                           static_cast<long long>(wide < tiles_x ? high : (at_once + tiles_x - 1) / tiles_x) * tile_tokens;
    if (!least || rows < least) least = rows, best = strips;
    if (static_cast<long long>(high) * high * tile_tokens < tile_rows) break;  // (flatter ones only need more)
  }
  const int rows = tiles_y > 1 ? tiles_y : shares, low = rows / best, tall = rows % best;  // (tall: how many strips are taller)
  *order = TileOrder{tiles_x, tiles_y, shares, best, in_turn, static_cast<int>(all), tiles_x * rows, low, tall * (low + 1), tall * (low + 1) * tiles_x,
                     divisor(tiles_x * rows), {divisor(tiles_x * low), divisor(tiles_x * (low + 1))}, {divisor(low), divisor(low + 1)}};
  return static_cast<unsigned>((in_turn ? (each + kDieUnits - 1) / kDieUnits * kDieUnits : each) * kDies);
}

// Weight rows and tokens that the tiles of each die would need, summed over the dies, with every eighth tile on a die; 0 where the dies could have
// rectangles of the grid of tiles.  No launch deals tiles out in either way: it is what wide_fetch() of gemm_wide.hip prices, and why is said there.
inline double big_operands(int tiles_x, int tiles_y, int tile_rows, int tile_tokens) {
  if (static_cast<long long>(tiles_x) * tiles_y >= 4 * kDies * kDieUnits) return 0.0;
  for (int dx = 1; dx <= kDies; dx *= 2)
    if (tiles_x % dx == 0 && tiles_y % (kDies / dx) == 0) return 0.0;
  const double tiles = static_cast<double>(tiles_x) * tiles_y, dies = tiles < kDies ? tiles : kDies, each = tiles / dies;
  const int columns = tiles_x / (tiles_x % 4 == 0 ? 4 : tiles_x % 2 == 0 ? 2 : 1);  // of tiles that a die meets
  return dies * ((each < columns ? each : columns) * tile_rows + (each < tiles_y ? each : tiles_y) * tile_tokens);
}

// Products of more than 64 tokens whose activations are 16-byte aligned with k % 8 == 0 (gemm_wide.hip).
int wide_splits(int n, int m, int k, int whole_bytes);
int wide_parts(int n, int m, int k, int gated);
int wide_tiles(int n, int m, int k, int gated, int ksplit);
void wide_tile_size(int tile, int* rows, int* tokens);
bool wide_serves(int lda, int k);
void wide_product(hipStream_t s, const bf16* a, int lda, int n, int k, const uint4* wt, int m, const float* bias, void* out,
                  int ldo, int out_f32, int accumulate, int gated, int ksplit);

// Up to 256 tokens n counts as the power of two above it: a choice made by it is then the same for every number
// of tokens that a captured decode step may stand for.
inline int counted_tokens(int n) {
  if (n > 256) return n;
  int tokens = 32;
  while (tokens < n) tokens *= 2;
  return tokens;
}

// plain_act()'s argument for the rows from `first` on
inline int plain_act_from(int accumulate, int first) {
  if (accumulate < kPlainSiluRows) return accumulate;
  const int left = accumulate / kPlainSiluRows - first;
  return left > 0 ? left * kPlainSiluRows : 0;
}

}  // namespace shk
