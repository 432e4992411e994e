// Products of up to 16 tokens, with small matrices of more (64, projections to heads 512), that finish what the kernels between
// two products would do, so that a decode step has fewer dependent kernels: five a layer instead of eight.  A step of a small model is a chain of kernels of 2.5 to 6 us each,
// most of which start, wait for memory once and end (weights already in the caches make the 7B output projection 6.3 us
// instead of 6.8).
//
// An output or down projection (few_stream) adds its result to the float32 residual stream and leaves the stream times
// the next norm's weight in bfloat16, with the sums of squares of every workgroup's rows beside it.  The product
// that reads those rows multiplies its sums by 1 / rms at the end: rsqrt(mean(x^2) + eps) is the same for a whole row,
// and W (x w) / rms = W (x w / rms).  So the norm between two products is no kernel of its own, and nobody waits for
// a row to be whole before multiplying.  (Forming the norm at the head of every workgroup of the next product was
// slower than the kernel it replaced.)
// A query/key/value projection (few_heads) rotates what it has formed and writes keys and values into their pages.
//
// Rows travel between these kernels as [k / 8][n][8]: sixteen neighbouring lanes of a matrix operand then read
// neighbouring pieces of 16 bytes, where rows of their own would cost a cache line a lane (896 x 4864 at 16 tokens 9.6 us,
// 7.8 so; 3584 x 18944 at 8 tokens 25.7, 23.2).
//
// Weights cold, chains of one kind of call, us at 1 / 8 / 16 tokens.  Product and norm against few_stream: 896 x 896
// 5.6 / 6.0 / 6.4 -> 2.9 / 3.0 / 3.0, 896 x 4864 6.9 / 7.3 / 7.5 -> 5.3 / 5.9 / 5.8, 3584 x 3584 9.6 / 9.5 / 10.4 -> 6.1 / 7.4 / 8.3,
// 3584 x 18944 26.4 / 26.7 / 29.6 -> 21.9 / 24.1 / 27.0.  Projections, rotation and cache write against few_heads: 1152 x 896
// 5.5 / 6.1 / 6.4 -> 4.1 / 4.3 / 4.4, 4608 x 3584 10.7 / 11.1 / 12.2 -> 10.4 / 11.2 / 12.3, 7168 x 5120 16.4 / 16.2 / 18.2 -> 14.2 / 15.4 /
// 17.2.  few_gated against the product without the division: 9728 x 896 5.6 / 6.2 / 6.9 -> 5.9 / 6.1 / 6.4, 37888 x 3584 40.6 /
// 40.6 / 45.1 -> 40.9 / 40.9 / 42.1.  Steps: 0.5B at 1 / 4 / 16 sequences 755 / 814 / 917 -> 653 / 692 / 757, 7B at 1 / 8 / 16
// 2,883 / 3,174 / 3,366 -> 2,686 / 3,000 / 3,158.
#include "gemm_few.h"

namespace shk {

// A workgroup takes NB blocks of 16 tokens; blockIdx.y says which.
template <int NB>
__device__ __forceinline__ int few_first() {
  return blockIdx.y * 16 * NB;
}

// Rows: piece `col` (a multiple of 8) of a token lies at token * token_step + col * col_step.
struct FewRows {
  const bf16* a;
  int token_step, col_step, n, k;
};

template <int NB>
struct FewTokens {
  const FewRows& x;
  __device__ __forceinline__ void operator()(const bf16* (&arow)[NB]) const {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int token = few_first<NB>() + b * 16 + static_cast<int>(threadIdx.x % 16);
      arow[b] = x.a + static_cast<size_t>(min(token, x.n - 1)) * x.token_step;
    }
  }
};

// What divides them: the squares' sums [count][n], null for rows that are normed already.
struct FewScale {
  const float* sums;
  int count;
  float inv_width, eps;
};

// A thread adds up some of the sums of one token.  They are asked for before the weights, all at once ...
template <int LOADS, int NB>
struct FewSquares {
  static constexpr int kTokens = 16 * NB;
  float v[LOADS > 0 ? LOADS : 1];
  __device__ __forceinline__ void load(const FewScale& s, int n) {
    const int token = few_first<NB>() + threadIdx.x % kTokens, first = threadIdx.x / kTokens, step = blockDim.x / kTokens;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int c = first + i * step;
      const float x = s.sums[static_cast<size_t>(c < s.count ? c : 0) * n + (token < n ? token : 0)];
      v[i] = c < s.count ? x : 0.f;
    }
  }
  // ... and left by wavefront while the weights travel
  __device__ __forceinline__ void leave(float* part) {
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) t += v[i];
#pragma unroll
    for (int off = kTokens; off < kWave; off <<= 1) t += __shfl_xor(t, off, kWave);
    if (threadIdx.x % kWave < kTokens) part[threadIdx.x / kWave * kTokens + threadIdx.x % kWave] = t;
  }
  __device__ __forceinline__ float scale(const FewScale& s, const float* part, int token, int waves) const {
    if (LOADS == 0) return 1.f;
    float t = 0.f;
    for (int w = 0; w < waves; ++w) t += part[w * kTokens + token];
    return rsqrtf(t * s.inv_width + s.eps);
  }
};

constexpr int kFewWaves = 9;  // wavefronts of a workgroup at most
constexpr int kFewHalfWaves = 4, kFewHalfTiles = 8;  // of one for half a block and 8 tokens; its tiles of a batch

// What a workgroup of few_stream's kernels does with the sum of weight row `row` and a token: it joins the stream, goes out times the next norm's
// weight, and its square with those of the ROWS rows beside it (neighbouring lanes) is their group's sum.
template <int ROWS>
__device__ __forceinline__ void few_join(float v, float w, int row, int token, bool mine, int n, int m, float* __restrict__ resid,
                                         bf16* __restrict__ rows, float* __restrict__ sums) {
  float square = v * v;
#pragma unroll
  for (int off = 1; off < ROWS; off <<= 1) square += __shfl_xor(square, off, kWave);
  if (!mine) return;
  resid[static_cast<size_t>(token) * m + row] = v;
  rows[(static_cast<size_t>(row / 8) * n + token) * 8 + row % 8] = from_float<bf16>(v * w);
  if (row % ROWS == 0) sums[static_cast<size_t>(row / ROWS) * n + token] = square;
}

// ROWS = 16: a workgroup for a block of 16 weight rows.  ROWS = 8: for half of one (a tile's pieces of 8 rows are whole
// lines of 128 bytes), where whole blocks leave compute units idle; the other half of the matrix instruction does the same again.
template <int C, int ROWS, int NB>
__global__ void __launch_bounds__(kFewWaves* kWave)
    few_stream_kernel(FewRows x, const u32x4* __restrict__ wt, int ktiles, int m, const float* __restrict__ bias,
                      float* __restrict__ resid, const float* __restrict__ weight, bf16* __restrict__ rows,
                      float* __restrict__ sums) {
  extern __shared__ f32x4 red[];  // [waves][NB][64]
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), waves = blockDim.x / kWave;
  const int wr = blockIdx.x * ROWS + lane % ROWS;
  const int inside = threadIdx.x / ROWS, r = threadIdx.x % ROWS, row = blockIdx.x * ROWS + r;
  float old[NB], w = 0.f;
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    const int token = few_first<NB>() + c * 16 + inside;
    old[c] = inside < 16 && token < x.n ? resid[static_cast<size_t>(token) * m + row] : 0.f;
  }
  if (inside < 16) {
    w = weight[row];
    if (bias) {
      const float add = bias[row];
#pragma unroll
      for (int c = 0; c < NB; ++c) old[c] += add;
    }
  }
  const u32x4* const wrow[1] = {wt + static_cast<size_t>(wr / 16) * ktiles * kWave + wr % 16 + lane / 16 * 16};
  f32x4 acc[1][NB];
  few_multiply<C, 4, 1, NB>(acc, wrow, FewTokens<NB>{x}, x.col_step, x.k, ktiles, wave, waves, [] {});
#pragma unroll
  for (int c = 0; c < NB; ++c) red[(wave * NB + c) * kWave + lane] = acc[0][c];
  __syncthreads();
  if (inside >= 16) return;
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    const int token = few_first<NB>() + c * 16 + inside;
    const float v = few_sum(red + c * kWave, NB * kWave, r, inside, waves) + old[c];
    few_join<ROWS>(v, w, row, token, token < x.n, x.n, m, resid, rows, sums);
  }
}

struct FewHalfTokens {  // the same 8 tokens for both halves of an operand
  const FewRows& x;
  __device__ __forceinline__ void operator()(const bf16* (&arow)[1]) const {
    arow[0] = x.a + static_cast<size_t>(min(static_cast<int>(blockIdx.y * 8 + threadIdx.x % 8), x.n - 1)) * x.token_step;
  }
};

// The same for half a block and 8 tokens.  The `walks` sums that a whole block's wavefronts form, each of every walks-th k-tile, go two to a
// wavefront: an operand of 16 rows holds these 8 of a tile of one walk and of a tile of the other, the tokens' operand 8 tokens of both, and two
// diagonal quarters of the results are the two sums (the others mix walks and are left).  So a row's bits are those that the kernel above gives.
// What bounds that one: a compute unit takes in 64 bytes a clock, half of them the same 8 rows again.  Chains with cold weights, us at 1 / 8 / 16
// tokens, above and here: 896 x 896 3.0 / 3.1 / 3.2 -> 2.9 / 3.0 / 3.0, 896 x 4864 6.0 / 6.1 / 7.0 -> 5.3 / 5.9 / 5.8, 1024 x 4096 5.6 / 5.7 / 6.0 -> 4.6 /
// 5.1 / 5.0, 2048 x 8192 at 1 / 8 11.1 / 11.1 -> 8.4 / 9.4.  Batches of 4, 12 or 16 tiles in place of 8: 896 x 4864 at one token 5.7, 5.8, 5.5.  (Two
// neighbouring tiles of one walk in an operand, which lets eight wavefronts share k: 4.9 / 5.6 / 6.7, but other sums than a whole block's.)
template <int C>
__global__ void __launch_bounds__(kFewHalfWaves* kWave)
    few_stream_half_kernel(FewRows x, const u32x4* __restrict__ wt, int ktiles, int m, const float* __restrict__ bias,
                           float* __restrict__ resid, const float* __restrict__ weight, bf16* __restrict__ rows,
                           float* __restrict__ sums, int walks) {
  extern __shared__ f32x4 red[];  // [waves][64]
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int inside = threadIdx.x / 8, r = threadIdx.x % 8, row = blockIdx.x * 8 + r, token = blockIdx.y * 8 + inside;
  const bool mine = inside < 8 && token < x.n;
  float old = mine ? resid[static_cast<size_t>(token) * m + row] : 0.f, w = 0.f;
  if (inside < 8) {
    w = weight[row];
    if (bias) old += bias[row];
  }
  const u32x4* const wrow[1] = {wt + static_cast<size_t>(blockIdx.x / 2) * ktiles * kWave + blockIdx.x % 2 * 8 + lane % 8 + lane / 16 * 16};
  const int walk = 2 * wave + lane % 16 / 8;  // (an odd number of them: the last one's neighbour is none, all zeros)
  f32x4 acc[1][1];
  few_multiply<C, kFewHalfTiles, 1, 1>(acc, wrow, FewHalfTokens{x}, x.col_step, x.k, ktiles, walk < walks ? walk : ktiles, walks, [] {});
  red[wave * kWave + lane] = acc[0][0];
  __syncthreads();
  if (inside >= 8) return;
  // element (r, token) of an even walk, (r + 8, token + 8) of an odd one, added in their order
  const float* p = reinterpret_cast<const float*>(red + r / 4 * 16 + inside) + r % 4;
  float v = 0.f;
  for (int t = 0; t < walks; ++t) v += p[(t / 2 * kWave + t % 2 * (2 * 16 + 8)) * 4];
  few_join<8>(v + old, w, row, token, mine, x.n, m, resid, rows, sums);
}

// A gated product: a workgroup for a gate block and its up block.
template <int C, int LOADS, int NB>
__global__ void __launch_bounds__(kFewWaves* kWave)
    few_gated_kernel(FewRows x, const u32x4* __restrict__ wt, int ktiles, int m, FewScale scaled, const float* __restrict__ args,
                     bf16* __restrict__ out, int ldo, int act) {
  extern __shared__ f32x4 red[];  // [waves][2][NB][64], then the squares' sums by wavefront [waves][16 NB]
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), waves = blockDim.x / kWave;
  float* part = reinterpret_cast<float*>(red + waves * 2 * NB * kWave);
  FewSquares<LOADS, NB> squares;
  squares.load(scaled, x.n);
  const u32x4* first = wt + static_cast<size_t>(blockIdx.x) * 2 * ktiles * kWave + lane;
  const u32x4* const wrow[2] = {first, first + static_cast<size_t>(ktiles) * kWave};
  f32x4 acc[2][NB];
  few_multiply<C, 2, 2, NB>(acc, wrow, FewTokens<NB>{x}, x.col_step, x.k, ktiles, wave, waves, [&] { squares.leave(part); });
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    red[(wave * 2 * NB + c) * kWave + lane] = acc[0][c];
    red[((wave * 2 + 1) * NB + c) * kWave + lane] = acc[1][c];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < NB * 256; e += blockDim.x) {
    const int inside = e / 16, token = few_first<NB>() + inside, r = e % 16, row = blockIdx.x * 16 + r;
    if (token >= x.n || row >= m) continue;
    const float s = squares.scale(scaled, part, inside, waves);
    const f32x4* mine = red + inside / 16 * kWave;
    const float g = few_sum(mine, 2 * NB * kWave, r, inside % 16, waves) * s;
    const float u = few_sum(mine + NB * kWave, 2 * NB * kWave, r, inside % 16, waves) * s;
    const size_t at = ldo ? static_cast<size_t>(token) * ldo + row : (static_cast<size_t>(row / 8) * x.n + token) * 8 + row % 8;
    out[at] = from_float<bf16>(gate_times_up(g, u, act, args));
  }
}

// Projections to queries, keys and values.  A workgroup forms 16 rows of the stacked matrix: of a query or key head 8 elements
// of the first half and their partners of the second, so that the rotation finds both, of the values 16 elements in a
// row.  The last wavefront multiplies nothing: it looks up pages and forms cosines and sines meanwhile.
template <int C, int LOADS>
__global__ void __launch_bounds__(kFewWaves* kWave)
    few_heads_kernel(FewRows x, const u32x4* __restrict__ wt, int ktiles, FewScale scaled, const float* __restrict__ bias,
                     bf16* __restrict__ out, int heads, int kv_heads, int head_dim, const float* __restrict__ inv_freq,
                     const int32_t* __restrict__ positions, const int32_t* __restrict__ token_seq,
                     const int32_t* __restrict__ tables, int table_stride, bf16* __restrict__ k_pool, bf16* __restrict__ v_pool,
                     int page_size, int num_pages, int write_kv, float magnitude) {
  extern __shared__ f32x4 red[];  // [waves][64], then the squares' sums by wavefront [waves + 1][16]
  __shared__ float cosine[16][8], sine[16][8];
  __shared__ int page_of[16], slot_of[16];
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), waves = blockDim.x / kWave - 1;
  float* part = reinterpret_cast<float*>(red + waves * kWave);
  const int per_head = head_dim / 16, head = blockIdx.x / per_head, group = blockIdx.x % per_head;
  const bool turned = head < heads + kv_heads;
  // this workgroup's first row and, eight rows on, where the other eight begin
  const int first = head * head_dim + group * (turned ? 8 : 16), second = first + (turned ? head_dim / 2 : 8);
  FewSquares<LOADS, 1> squares;
  squares.load(scaled, x.n);
  if (wave == waves) {
    if (LOADS) squares.leave(part);
    if (lane < 16 && few_first<1>() + lane < x.n) {
      const int pos = positions[few_first<1>() + lane];
      int page = -1;
      if (write_kv && head >= heads)
        page = tables[static_cast<size_t>(token_seq[few_first<1>() + lane]) * table_stride + pos / page_size];
      page_of[lane] = page >= 0 && page < num_pages ? page : -1;  // (outside: a host bug; never dereferenced)
      slot_of[lane] = pos % page_size;
    }
    if (turned) {
#pragma unroll
      for (int e = lane; e < 128; e += kWave) {  // (angles as in rope_kv.hip)
        const int token = min(few_first<1>() + e / 8, x.n - 1);
        const float angle = static_cast<float>(positions[token]) * inv_freq[group * 8 + e % 8];
        const double wide = static_cast<double>(angle);
        const double turns = rint(wide * 0.15915494309189535);
        const float reduced = static_cast<float>(fma(turns, -6.283185307179586, wide));
        float sv, cv;
        sincosf(reduced, &sv, &cv);
        cosine[e / 8][e % 8] = cv * magnitude;
        sine[e / 8][e % 8] = sv * magnitude;
      }
    }
  } else {
    const int wr = lane % 16 < 8 ? first + lane % 16 : second + lane % 16 - 8;
    const u32x4* const wrow[1] = {wt + static_cast<size_t>(wr / 16) * ktiles * kWave + wr % 16 + lane / 16 * 16};
    f32x4 acc[1][1];
    few_multiply<C, 4, 1, 1>(acc, wrow, FewTokens<1>{x}, x.col_step, x.k, ktiles, wave, waves, [&] { if (LOADS) squares.leave(part); });
    red[wave * kWave + lane] = acc[0][0];
  }
  const int inside = threadIdx.x / 8, token = few_first<1>() + inside, i = threadIdx.x % 8;
  float b1 = 0.f, b2 = 0.f;
  if (bias) b1 = bias[first + i], b2 = bias[second + i];
  __syncthreads();
  if (inside >= 16 || token >= x.n) return;
  const float s = squares.scale(scaled, part, inside, waves + 1);
  const float x1 = few_sum(red, kWave, i, inside, waves) * s + b1, x2 = few_sum(red, kWave, i + 8, inside, waves) * s + b2;
  const float c = turned ? cosine[inside][i] : 1.f, t = turned ? sine[inside][i] : 0.f;
  const float o1 = turned ? x1 * c - x2 * t : x1, o2 = turned ? x2 * c + x1 * t : x2;
  if (head < heads) {
    bf16* row = out + static_cast<size_t>(token) * (heads + 2 * kv_heads) * head_dim;
    row[first + i] = from_float<bf16>(o1);
    row[second + i] = from_float<bf16>(o2);
    return;
  }
  if (page_of[inside] < 0) return;
  const int kv = turned ? head - heads : head - heads - kv_heads;
  const size_t base = (static_cast<size_t>(page_of[inside]) * kv_heads + kv) * page_size * head_dim;
  const int slot = slot_of[inside], e1 = first - head * head_dim + i, e2 = second - head * head_dim + i;
  if (turned) {
    k_pool[base + key_offset(slot, e1, page_size, head_dim)] = from_float<bf16>(o1);
    k_pool[base + key_offset(slot, e2, page_size, head_dim)] = from_float<bf16>(o2);
  } else {
    v_pool[base + static_cast<size_t>(e1) * page_size + slot] = from_float<bf16>(o1);
    v_pool[base + static_cast<size_t>(e2) * page_size + slot] = from_float<bf16>(o2);
  }
}

}  // namespace shk

using namespace shk;

constexpr int kFewTokens = 64, kFewHeadsTokens = 512;

static bool few_rows_of(FewRows* x, const void* a, int lda, int n, int k, int most) {
  const bool pieces = lda == 0;  // [k / 8][n][8]
  *x = FewRows{static_cast<const bf16*>(a), pieces ? 8 : lda, pieces ? n : 1, n, k};
  return n >= 0 && n <= most && k > 0 && k % 8 == 0 && (pieces || (lda >= k && lda % 8 == 0));
}

// fn with the loads of a thread that adds up squares (at least one) as a constant
template <typename Fn>
static void with_loads(int count, int threads, Fn fn) {
  const int loads = (count + threads / 16 - 1) / (threads / 16);
  if (loads <= 4) fn(std::integral_constant<int, 4>{});
  else if (loads <= 8) fn(std::integral_constant<int, 8>{});
  else fn(std::integral_constant<int, 16>{});
}
constexpr int kFewMostLoads = 16;

// Half blocks where whole ones would be one for every second compute unit or fewer: 896 x 4864 at 8 tokens 6.6 us whole, 5.9 in
// halves, 2048 x 11008 12.7 and 11.8; 3584 x 18944 23.2 and 32.1.
static int few_stream_rows(int m) { return m <= 2048 ? 8 : 16; }

// Half blocks of 8 tokens, whose wavefronts take two walks of k each: up to 8 tokens, and as long as all of them are at work at once.  At 16 / 32
// tokens in blocks of 16 and of 8: 896 x 4864 7.0 / 6.6 and 5.8 / 8.9 us, 512 x 2048 4.1 / 4.0 and 3.4 / 3.5, 1536 x 1536 4.0 / 5.0 and 4.3 / 5.2.
static bool few_stream_paired(int n, int m) { return n <= 8 || (n + 7LL) / 8 * (m / 8) <= kDies * kDieUnits; }

// The most rows * k for which 17 to 64 tokens go this way: every 16 of them read the weights again, from the caches.
// At 17 / 32 / 64 tokens, with the norm: 896 x 896 7.6 / 7.6 / 7.6 -> 3.6 / 3.6 / 4.7, 896 x 4864 10.3 / 11.0 / 12.2 -> 6.3 / 6.6 / 9.5,
// but 1536 x 8960 12.7 / 13.5 / 16.9 -> 17.5 / 18.6 / 26.6.  Heads, with the position kernel: 1152 x 896 7.7 / 7.7 / 7.8 -> 4.4 / 4.6 /
// 5.3, 2560 x 2048 9.9 / 11.1 / 14.0 -> 9.2 / 9.7 / 13.3, 4608 x 3584 13.7 / 14.4 / 18.1 -> 16.9 / 17.8 / 29.  Gated, without the norm
// that it spares: 9728 x 896 7.2 / 7.4 / 10.0 -> 7.5 / 7.9 / 10.4, 17920 x 1536 12.9 / 13.5 / 16.8 -> 13.7 / 15.0 / 23.2.
constexpr long long kFewStreamMost = 5 * 1000 * 1000, kFewHeadsMost = 6 * 1000 * 1000, kFewGatedMost = 10 * 1000 * 1000;

// Heads of more tokens, which spare the position kernel of so many rows: as long as what all blocks of 16 tokens read together
// stays below this.  Cold weights, product and position kernel against this, at 65 / 128 / 256 / 384 / 512 tokens: 512 x 256
// 9.1 / 9.2 / 9.4 / 9.4 / 9.7 -> 3.2 / 3.6 / 4.0 / 4.4 / 4.7 us, 1152 x 896 9.9 / 10.0 / 12.2 / 12.5 / 13.4 -> 5.3 / 6.6 / 8.8 /
// 11.8 / 14.4 (the line lies at 400), 2048 x 1536 12.3 / 13.3 / 18.5 -> 9.2 / 12.7 / 20.6 (at 128), 2560 x 2048 15.7 / 16.8 -> 14.0 / 20.7.
constexpr long long kFewHeadsRead = 26 * 1000 * 1000;
// Of 17 to 64 tokens, whose product's own kernel reads the weights once, at 17 / 32: 4608 x 1536 11.6 / 13.3 -> 11.5 / 12.3, 3584 x 2560 11.9 /
// 13.6 -> 11.7 / 12.0, 4096 x 2304 11.6 / 12.8 -> 11.0 / 11.6, but 4096 x 2560 11.9 / 13.3 -> 12.3 / 12.7, 4608 x 2304 11.8 / 13.0 -> 13.7 / 14.5,
// 6144 x 2048 12.9 / 13.9 -> 15.2 / 15.6.
constexpr long long kFewHeadsReadFew = 20 * 1000 * 1000;

static bool few_takes(int n, int m, int k, long long most) {
  return n <= 16 || (n <= kFewTokens && static_cast<long long>(m) * k <= most);
}

// Not where a second round of workgroups would be nearly empty: 320 of them (5120 x 5120 at 8 tokens 14.3 us for product in shares
// and norm, 15.1 here; 5120 x 13824 28.0 and 31.4).  256 are a round: 4096 x 14336 23.7 -> 20.0.
// Nor where few workgroups walk a long k, which shares of it spread over the chip.  Product and norm against this at 1 / 8 / 16 tokens: 1024 x 5120
// 7.3 / 7.3 / 7.9 -> 5.7 / 6.2 / 6.0, 512 x 8192 7.6 / 8.1 / 8.4 -> 6.4 / 7.3 / 7.1, 256 x 18944 8.3 / 8.7 / 9.1 -> 11.8 / 13.5 / 13.1, 1536 x 6144 10.4 /
// 11.0 / 11.1 -> 6.5 / 7.5 / 8.7, x 8960 10.1 / 10.9 / 13.2 -> 8.7 / 10.9 / 12.4, x 18944 15.1 / 17.0 / 21.7 -> 15.2 / 18.5 / 22.7, 2048 x 8192 11.4 / 11.8 /
// 12.7 -> 8.4 / 9.4 / 11.7, x 14336 15.7 / 16.4 / 17.6 -> 12.8 / 14.5 / 19.6; whole blocks, 2304 x 9216 12.3 / 13.2 / 14.5 -> 12.5 / 13.6 / 15.9, 2560 x 8192
// 12.1 / 12.1 / 13.1 -> 11.5 / 10.8 / 12.7, x 13824 16.3 / 15.8 / 17.7 -> 17.6 / 16.3 / 19.3; 192 workgroups and more at any k: 3072 x 18944 23.9 / 24.8 / 27.7 -> 23.0 /
// 22.4 / 26.3, 4096 x 24576 36.3 / 37.8 / 41.0 -> 33.9 / 32.7 / 35.9; 64 tokens, 256 x 6144 8.6 -> 10.0, 512 x 5120 10.6 -> 9.4, x 8192 11.0 -> 12.8.
// (Half blocks' line was drawn while a wavefront took one walk, 512 x 8192 8.7 / 8.8 / 9.4, 1536 x 8960 11.5 / 11.5 / 11.6, 2048 x 14336 17.9 / 15.0 / 16.3.  It
// stands there, so that the sizes between keep the order in which shares and norm add them up.)
extern "C" int shk_few_stream_sums(int n, int m, int k) {
  const bool near = m >= 3072 || k <= 5120 || (m <= 2048 ? k <= 4 * m : 2 * k <= 7 * m);
  return m > 0 && m <= 4096 && m % 16 == 0 && k > 0 && k % 8 == 0 && near && few_takes(n, m, k, kFewStreamMost) ? m / few_stream_rows(m) : 0;
}

// `m` rows of the gate and as many of the other matrix; the k columns may come with as many sums as few_stream leaves.
extern "C" int shk_few_gated_takes(int n, int m, int k) { return m > 0 && k > 0 && k % 8 == 0 && few_takes(n, 2 * m, k, kFewGatedMost); }

extern "C" int shk_few_heads_takes(int n, int m, int k) {
  if (m <= 0 || k <= 0 || k % 8) return 0;
  if (few_takes(n, m, k, kFewHeadsMost)) return 1;
  return n <= kFewHeadsTokens && (counted_tokens(n) + 15LL) / 16 * m * k <= (n <= kFewTokens ? kFewHeadsReadFew : kFewHeadsRead);
}

extern "C" int shk_few_stream(const void* a, int lda, int n, int k, const void* wt, int m, const float* bias, float* resid,
                              const float* weight, void* rows, float* sums, void* stream) {
  FewRows x;
  SHK_REQUIRE(few_rows_of(&x, a, lda, n, k, kFewTokens) && m > 0 && m % 16 == 0, "few_stream: bad sizes n=%d m=%d k=%d lda=%d", n, m, k, lda);
  if (n == 0) return 0;
  SHK_REQUIRE(a && wt && resid && weight && rows && sums, "few_stream: null pointer");
  SHK_REQUIRE(reinterpret_cast<uintptr_t>(a) % 16 == 0, "few_stream: rows are not 16-byte aligned");
  const int kt = (k + 31) / 32, waves = few_waves(kt, kFewTiles), rows_each = few_stream_rows(m);
  with_tiles<kFewTiles>((kt + waves - 1) / waves, [&](auto c) {
    const auto go = [&](auto kernel, int tokens, int wavefronts, auto... more) {
      kernel<<<dim3(m / rows_each, (n + tokens - 1) / tokens), wavefronts * kWave, (tokens + 15) / 16 * wavefronts * kWave * sizeof(f32x4), static_cast<hipStream_t>(stream)>>>(
          x, static_cast<const u32x4*>(wt), kt, m, bias, resid, weight, static_cast<bf16*>(rows), sums, more...);
    };
    if (rows_each == 16) return go(few_stream_kernel<c.value, 16, 1>, 16, waves);
    if (few_stream_paired(n, m)) return go(few_stream_half_kernel<c.value>, 8, (waves + 1) / 2, waves);
    if constexpr (c.value == 0) {
      // two blocks of tokens in a workgroup where many tokens would have a long k read four times over (896 x 4864 at 64
      // tokens 10.4 us in one, 9.5; at 32 6.6 in one, 10.0)
      if (n > 32) return go(few_stream_kernel<0, 8, 2>, 32, waves);
    }
    go(few_stream_kernel<c.value, 8, 1>, 16, waves);
  });
  SHK_LAUNCH_CHECK("few_stream");
  return 0;
}

extern "C" int shk_few_gated(const void* a, int lda, int n, int k, const void* wt, const float* sums, int count, float eps,
                             const float* args, void* out, int m, int ldo, int gated, void* stream) {
  FewRows x;
  SHK_REQUIRE(few_rows_of(&x, a, lda, n, k, kFewTokens) && m > 0 && (ldo ? ldo >= m : m % 8 == 0),
              "few_gated: bad sizes n=%d m=%d k=%d lda=%d ldo=%d", n, m, k, lda, ldo);
  SHK_REQUIRE(gated > 0 && gated <= kActQuickGelu, "few_gated: unknown gate activation %d", gated);
  SHK_REQUIRE(sums && count > 0 && eps > 0.f, "few_gated: rows come with the sums of their squares");
  if (n == 0) return 0;
  SHK_REQUIRE(a && wt && out, "few_gated: null pointer");
  SHK_REQUIRE(reinterpret_cast<uintptr_t>(a) % 16 == 0, "few_gated: rows are not 16-byte aligned");
  const FewScale scaled = {sums, count, 1.f / static_cast<float>(k), eps};
  // four wavefronts where they hold their tiles at once (9728 x 896: 5.8 us with one token, 5.9 in eight), else eight
  // (22016 x 2048 15.6, 15.9 in four)
  const int kt = (k + 31) / 32, waves = kt <= 4 * kFewPairs ? 4 : 8;
  SHK_REQUIRE(count <= kFewMostLoads * waves * 4 / (n > 16 ? 2 : 1), "few_gated: too many sums (%d)", count);
  const int nb = n > 16 ? 2 : 1;  // (9728 x 896 at 17 / 32 / 64 tokens 8.2 / 8.5 / 12.4 us in one, 7.5 / 7.9 / 10.4)
  with_loads(count, waves * kWave / nb, [&](auto loads) {
    with_tiles<kFewPairs>((kt + waves - 1) / waves, [&](auto c) {
      const size_t lds = nb * waves * (2 * kWave * sizeof(f32x4) + 16 * sizeof(float));
      const auto kernel = nb == 2 ? few_gated_kernel<c.value, loads.value, 2> : few_gated_kernel<c.value, loads.value, 1>;
      kernel<<<dim3((m + 15) / 16, (n + 16 * nb - 1) / (16 * nb)), waves * kWave, lds, static_cast<hipStream_t>(stream)>>>(
          x, static_cast<const u32x4*>(wt), kt, m, scaled, args, static_cast<bf16*>(out), ldo, gated);
    });
  });
  SHK_LAUNCH_CHECK("few_gated");
  return 0;
}

extern "C" int shk_few_heads(const void* a, int lda, int n, int k, const void* wt, const float* sums, int count, float eps,
                             const float* bias, void* out, int heads, int kv_heads, int head_dim, const float* inv_freq,
                             const int32_t* positions, const int32_t* token_seq, const int32_t* tables, int table_stride,
                             void* k_pool, void* v_pool, int page_size, int num_pages, int write_kv, float magnitude,
                             void* stream) {
  FewRows x;
  SHK_REQUIRE(few_rows_of(&x, a, lda, n, k, kFewHeadsTokens), "few_heads: bad sizes n=%d k=%d lda=%d", n, k, lda);
  SHK_REQUIRE(heads > 0 && kv_heads > 0 && head_dim > 0 && head_dim % 16 == 0, "few_heads: bad heads %d %d %d", heads, kv_heads, head_dim);
  if (n == 0) return 0;
  SHK_REQUIRE(a && wt && out && inv_freq && positions, "few_heads: null pointer");
  SHK_REQUIRE(reinterpret_cast<uintptr_t>(a) % 16 == 0, "few_heads: rows are not 16-byte aligned");
  SHK_REQUIRE(!sums || (count > 0 && eps > 0.f), "few_heads: bad sums");
  if (write_kv) {
    SHK_REQUIRE(token_seq && tables && k_pool && v_pool, "few_heads: null cache pointer");
    SHK_REQUIRE(page_size > 0 && num_pages > 0 && table_stride > 0, "few_heads: bad cache sizes page_size=%d num_pages=%d table_stride=%d",
                page_size, num_pages, table_stride);
  }
  const FewScale scaled = {sums, count, 1.f / static_cast<float>(k), eps};
  const int groups = (heads + 2 * kv_heads) * (head_dim / 16);
  const int kt = (k + 31) / 32, waves = few_waves(kt, kFewTiles);
  SHK_REQUIRE(!sums || count <= kFewMostLoads * (waves + 1) * 4, "few_heads: too many sums (%d)", count);
  const auto go = [&](auto loads) {
    with_tiles<kFewTiles>((kt + waves - 1) / waves, [&](auto c) {
      const size_t lds = waves * kWave * sizeof(f32x4) + (waves + 1) * 16 * sizeof(float);
      few_heads_kernel<c.value, loads.value><<<dim3(groups, (n + 15) / 16), (waves + 1) * kWave, lds, static_cast<hipStream_t>(stream)>>>(
          x, static_cast<const u32x4*>(wt), kt, scaled, bias, static_cast<bf16*>(out), heads, kv_heads, head_dim, inv_freq, positions,
          token_seq, tables, table_stride, static_cast<bf16*>(k_pool), static_cast<bf16*>(v_pool), page_size, num_pages, write_kv,
          magnitude);
    });
  };
  if (sums)
    with_loads(count, (waves + 1) * kWave, go);
  else
    go(std::integral_constant<int, 0>{});
  SHK_LAUNCH_CHECK("few_heads");
  return 0;
}
