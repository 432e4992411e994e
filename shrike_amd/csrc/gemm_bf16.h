// What the kernels of bfloat16 products share: operand types, activations in their epilogues, and the order in which
// the large ones take their tiles.
#pragma once

#include "api.h"
#include "common.h"

namespace shk {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
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

// The tile of a workgroup of the large kernels; false: none (the grid is padded).
__device__ __forceinline__ bool big_tile(int tiles_x, int tiles_y, int by_die, int& tile_x, int& tile_y) {
  // Which tile: workgroups are handed to the chip's eight dies (each with its own
  // L2) in turn, workgroup p to die p % 8.  The tiles are therefore dealt out in
  // blocks of 32 (up to 8 token tiles of 32 / that many weight tiles) and block B goes to
  // die B % 8, whose 32 compute units then work on tiles that share their
  // operands: the die's L2 serves most of their loads.
  // With fewer tiles (by_die == 2 * dx) the grid of tiles is cut into dx x 8/dx
  // rectangles, one for each die, where the numbers of tiles allow that; else
  // (by_die == 0) the tiles are taken in plain order.
  tile_x = blockIdx.x % tiles_x, tile_y = blockIdx.x / tiles_x;
  if (by_die > 1) {
    const int die = blockIdx.x % kDies, turn = blockIdx.x / kDies;
    const int dx = by_die / 2, wide = tiles_x / dx, high = tiles_y / (kDies / dx);
    tile_x = (die % dx) * wide + turn % wide;
    tile_y = (die / dx) * high + turn / wide;
  } else if (by_die) {
    const int die = blockIdx.x % kDies, turn = blockIdx.x / kDies;
    const int block_y = tiles_y < 8 ? tiles_y : 8, block_x = kDieUnits / block_y;
    const int blocks_x = (tiles_x + block_x - 1) / block_x;
    const int block = (turn / kDieUnits) * kDies + die, within = turn % kDieUnits;
    tile_x = (block % blocks_x) * block_x + within / block_y;
    tile_y = (block / blocks_x) * block_y + within % block_y;
    if (within >= block_x * block_y) return false;
  }
  return tile_x < tiles_x && tile_y < tiles_y;
}

// The grid of the large kernels: how big_tile() is to deal out the tiles, and the number of workgroups.
inline unsigned big_grid(int tiles_x, int tiles_y, int tile_rows, int tile_tokens, int* by_die) {
  // one-dimensional, in whole rounds of the eight dies' blocks of 32 tiles
  const int block_y = tiles_y < 8 ? tiles_y : 8, block_x = kDieUnits / block_y;
  const long long blocks = static_cast<long long>((tiles_x + block_x - 1) / block_x) * ((tiles_y + block_y - 1) / block_y);
  // worth it from four rounds of workgroups on: below that, whole dies would stay idle
  *by_die = static_cast<long long>(tiles_x) * tiles_y >= 4 * kDies * kDieUnits;
  if (*by_die) return static_cast<unsigned>((blocks + kDies - 1) / kDies * kDies * kDieUnits);
  // one rectangle of tiles per die, cut so that a die's tiles share the most
  // operands (the fewest rows of weights and activations to read per die)
  long long least = 0;
  for (int dx = 1; dx <= kDies; dx *= 2) {
    const int dy = kDies / dx;
    if (tiles_x % dx || tiles_y % dy) continue;
    const long long rows = static_cast<long long>(tiles_x / dx) * tile_rows + static_cast<long long>(tiles_y / dy) * tile_tokens;
    if (!least || rows < least) least = rows, *by_die = 2 * dx;
  }
  return static_cast<unsigned>(tiles_x * tiles_y);
}

// Weight rows and tokens that the tiles of each die need, summed over the dies, where the tiles are taken in plain order (every
// eighth one on a die); 0 in the other orders, whose dies share.
inline double big_operands(int tiles_x, int tiles_y, int tile_rows, int tile_tokens) {
  int by_die;
  big_grid(tiles_x, tiles_y, tile_rows, tile_tokens, &by_die);
  if (by_die) return 0.0;
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
