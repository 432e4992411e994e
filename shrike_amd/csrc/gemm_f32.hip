// out[n, m] = a[n, k] @ w[m, k]^T + bias in float32 on the matrix units
// (v_mfma_f32_16x16x4_f32: products and sums of 24-bit mantissas, no reduced precision).
//
// Every product of the float32 mode goes through gemm_f32_kernel, whatever its number of rows, and
// a float32 result must have the same bits however a prompt is cut and whatever else is in the
// step.  So the order of the sum is a function of k alone and every shape of the kernel keeps it:
//   k is cut into at most 16 segments of L = 16 * ceil(k / 256) elements; within a segment the
//   matrix instruction walks k in steps of 16, instruction j = 0..3 of a step taking the elements
//   j, 4 + j, 8 + j, 12 + j (so that a lane's four operands are one 16-byte load of either
//   row-major matrix); segments 4g .. 4g + 3 are added in order to a group's sum, the four groups
//   in order to the result.
// What differs between shapes is which wavefront walks which segments: all 16 wavefronts of a
// workgroup one each (few rows: a chain of k is then k / 16 long, and 16 KiB of weights are in
// flight per workgroup), four a group each with 64 x 64 results per workgroup (many rows), or every one all
// of them (many rows and a k of up to 256).
// Operands go straight from memory to registers: an instruction takes 32 cycles of its SIMD, a 2 x 2
// arrangement of tiles needs 4 KiB of operands every 512 cycles and SIMD, which L1 and L2 deliver.
// The model's weights are held in tiles of 16 rows x 16 k (retile_f32_kernel): a wavefront's load is
// then one run of 1 KiB instead of 16 pieces of 64 bytes (four rows of a 9728 x 896 matrix 10.7 us
// against 14, of 896 x 4864 13 against 18).  Operands of other callers are row-major.
// What bounds it: with few rows the latency of one round of loads and a reduction through LDS; with
// many the supply of operands and the last round of workgroups, which leave half of the matrix instruction's rate
// (150 TFLOP/s alone; 9728 x 896 at 509 rows 75): a workgroup's wavefronts walk different parts of k and so share no operand,
// and loads are one step ahead.  At the full rate that would be 38 GB/s a compute unit, about what one takes in.  Before, one workgroup per 64 x 64 results with vector
// instructions: a 0.5B decode step of four requests 23.9 ms (2.4 with this kernel, 1.56 with attention_f32.hip as
// well), a 509-token prompt 42.6 ms (18.9, 6.5); the logits' error against 64 bits 6.4e-7 (2.5e-7).
#include "api.h"
#include "common.h"

namespace shk {

typedef float mf4 __attribute__((ext_vector_type(4)));

constexpr int kF32Segments = 16, kF32Group = 4;
constexpr int kDies = 8;

// Four consecutive k of one row.  VEC: k and the rows are multiples of 16 bytes.
template <bool VEC>
__device__ __forceinline__ mf4 load_k4(const float* __restrict__ row, int kk) {
  if (VEC) return *reinterpret_cast<const mf4*>(row + kk);
  return mf4{row[kk], row[kk + 1], row[kk + 2], row[kk + 3]};
}

// The same where the row ends at k: zeros beyond it.
__device__ __forceinline__ mf4 load_k4_end(const float* __restrict__ row, int kk, int k) {
  mf4 v;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float x = row[kk + j < k ? kk + j : 0];
    v[j] = kk + j < k ? x : 0.f;
  }
  return v;
}

// A wavefront forms RT x CT tiles of 16 features x 16 rows of a; a workgroup has KW wavefronts along k
// times MW x NW side by side.  U: steps of 16 of k that are loaded at once, ahead of their use.
template <int RT, int CT, int KW, int MW, int NW, int U, bool TILED, bool VEC>
__global__ void __launch_bounds__(kWave * KW * MW * NW)
    gemm_f32_kernel(const float* __restrict__ a, const float* __restrict__ w, const float* __restrict__ bias,
                    float* __restrict__ out, int n, int m, int k, int lda, int ldo, int accumulate, int vec_out,
                    long long a_batch, long long w_batch, long long out_batch) {
  constexpr int kTiles = MW * NW * RT * CT, kWaves = KW * MW * NW;
  __shared__ mf4 sums[KW][kTiles][kWave];
  a += blockIdx.z * a_batch;
  w += blockIdx.z * w_batch;
  out += blockIdx.z * out_batch;
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int kw = wave / (MW * NW), side = wave % (MW * NW), mw = side / NW, nw = side % NW;
  const int i = lane % 16, kg = lane / 16;
  // workgroup -> tile: each of the eight dies takes a run of tiles, the rows of a innermost, so that
  // a die reads its features' weights from memory once and finds them in its own L2 afterwards
  const int rows = (n + 16 * CT * NW - 1) / (16 * CT * NW), cols = (m + 16 * RT * MW - 1) / (16 * RT * MW);
  const int per_die = (rows * cols + kDies - 1) / kDies;
  const int tile = blockIdx.x % kDies * per_die + blockIdx.x / kDies;
  if (blockIdx.x / kDies >= per_die || tile >= rows * cols) return;
  const int bx = tile / rows, by = tile % rows;
  const int f0 = (bx * MW + mw) * RT * 16, t0 = (by * NW + nw) * CT * 16;

  // rows beyond the last are read as the last and not stored
  const float* wr[RT];
  const float* ar[CT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
    wr[r] = TILED ? w + static_cast<size_t>(min(f0 / 16 + r, (m - 1) / 16)) * ((k + 15) / 16) * 256 + lane * 4
                  : w + static_cast<size_t>(min(f0 + r * 16 + i, m - 1)) * k;
#pragma unroll
  for (int c = 0; c < CT; ++c) ar[c] = a + static_cast<size_t>(min(t0 + c * 16 + i, n - 1)) * lda;

  const int seg_steps = (k + 16 * kF32Segments - 1) / (16 * kF32Segments);
  constexpr int kMine = kF32Segments / KW;  // segments of this wavefront, side by side
  const int begin = min(kw * kMine * seg_steps * 16, k), end = min(begin + kMine * seg_steps * 16, k);
  const int steps = (end - begin) / 16;  // whole ones; only the matrix's last segment can end within one

  mf4 acc[RT][CT], group[RT][CT], total[RT][CT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[r][c] = group[r][c] = total[r][c] = mf4{0.f, 0.f, 0.f, 0.f};

  int in_seg = 0, in_group = 0;
  auto multiply = [&](const mf4(&wv)[RT], const mf4(&av)[CT]) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int c = 0; c < CT; ++c)
          acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[r][j], av[c][j], acc[r][c], 0, 0, 0);
    if (kMine > 1 && ++in_seg == seg_steps) {  // a segment ends
      in_seg = 0;
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int c = 0; c < CT; ++c) {
          group[r][c] += acc[r][c];
          acc[r][c] = mf4{0.f, 0.f, 0.f, 0.f};
        }
      if (kMine > kF32Group && ++in_group == kF32Group) {
        in_group = 0;
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int c = 0; c < CT; ++c) {
            total[r][c] += group[r][c];
            group[r][c] = mf4{0.f, 0.f, 0.f, 0.f};
          }
      }
    }
  };
  if (steps > 0) {
    mf4 wv[2][U][RT], av[2][U][CT];
    auto load = [&](int set, int s0) {
#pragma unroll
      for (int u = 0; u < U; ++u) {  // (unconditional loads: a step beyond the last is the last again)
        const int k0 = begin + min(s0 + u, steps - 1) * 16, kk = k0 + kg * 4;
#pragma unroll
        for (int r = 0; r < RT; ++r)
          wv[set][u][r] = TILED ? *reinterpret_cast<const mf4*>(wr[r] + static_cast<size_t>(k0) * 16) : load_k4<VEC>(wr[r], kk);
#pragma unroll
        for (int c = 0; c < CT; ++c) av[set][u][c] = load_k4<VEC>(ar[c], kk);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    load(0, 0);
    for (int s = 0; s < steps; s += 2 * U) {
      load(1, s + U);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (s + u < steps) multiply(wv[0][u], av[0][u]);
      load(0, s + 2 * U);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (s + U + u < steps) multiply(wv[1][u], av[1][u]);
    }
  }
  if (begin + steps * 16 < end) {
    mf4 wv[RT], av[CT];
    const int k0 = begin + steps * 16, kk = k0 + kg * 4;
#pragma unroll
    for (int r = 0; r < RT; ++r)
      wv[r] = TILED ? *reinterpret_cast<const mf4*>(wr[r] + static_cast<size_t>(k0) * 16) : load_k4_end(wr[r], kk, k);
#pragma unroll
    for (int c = 0; c < CT; ++c) av[c] = load_k4_end(ar[c], kk, k);
    multiply(wv, av);
  }

  // the open segment and group, then the wavefronts' shares in order
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      mf4 v = acc[r][c];
      if (kMine > 1) v = group[r][c] + v;
      if (kMine > kF32Group) v = total[r][c] + v;
      sums[kw][(side * RT + r) * CT + c][lane] = v;
    }
  __syncthreads();
  for (int t = wave; t < kTiles; t += kWaves) {
    mf4 v = mf4{0.f, 0.f, 0.f, 0.f};
    if (KW > kF32Segments / kF32Group) {
#pragma unroll
      for (int g = 0; g < KW; g += KW / 4) {
        mf4 s = mf4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int x = 0; x < KW / 4; ++x) s += sums[g + x][t][lane];
        v += s;
      }
    } else {
#pragma unroll
      for (int x = 0; x < KW; ++x) v += sums[x][t][lane];
    }
    const int s = t / (RT * CT), r = t / CT % RT, c = t % CT;
    const int row = ((by * NW + s % NW) * CT + c) * 16 + i;  // the matrix instruction's columns
    const int col = ((bx * MW + s / NW) * RT + r) * 16 + kg * 4;
    if (row >= n) continue;
    float* dst = out + static_cast<size_t>(row) * ldo + col;
    if (vec_out && col + 3 < m) {
      if (bias) v += mf4{bias[col], bias[col + 1], bias[col + 2], bias[col + 3]};
      if (accumulate) v += *reinterpret_cast<const mf4*>(dst);
      *reinterpret_cast<mf4*>(dst) = v;
      continue;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (col + e >= m) continue;
      float x = v[e];
      if (bias) x += bias[col + e];
      if (accumulate) x += dst[e];
      dst[e] = x;
    }
  }
}

struct F32Product {
  const float *a, *w, *bias;
  float* out;
  int n, m, k, lda, ldo, accumulate, batch;
  long long a_batch, w_batch, out_batch;
};

template <int RT, int CT, int KW, int MW, int NW, int U, bool TILED>
static void launch_f32(const F32Product& p, hipStream_t s) {
  constexpr int F = 16 * RT * MW, T = 16 * CT * NW;
  const int tiles = (p.m + F - 1) / F * ((p.n + T - 1) / T);
  const dim3 grid((tiles + kDies - 1) / kDies * kDies, 1, p.batch);
  bool vec = p.lda % 4 == 0 && p.a_batch % 4 == 0 && reinterpret_cast<uintptr_t>(p.a) % 16 == 0;
  if (!TILED) vec = vec && p.k % 4 == 0 && p.w_batch % 4 == 0 && reinterpret_cast<uintptr_t>(p.w) % 16 == 0;
  const int vec_out = p.ldo % 4 == 0 && p.out_batch % 4 == 0 && reinterpret_cast<uintptr_t>(p.out) % 16 == 0;
  auto kernel = vec ? gemm_f32_kernel<RT, CT, KW, MW, NW, U, TILED, true> : gemm_f32_kernel<RT, CT, KW, MW, NW, U, TILED, false>;
  kernel<<<grid, kWave * KW * MW * NW, 0, s>>>(p.a, p.w, p.bias, p.out, p.n, p.m, p.k, p.lda, p.ldo, p.accumulate, vec_out,
                                               p.a_batch, p.w_batch, p.out_batch);
}

// The shape of the kernel for a size (results are the same bits in all of them).  Measured on the 0.5B
// model's matrices, tiled weights, microseconds:
//   up to 16 rows: 896 x 896 5 in one-tile workgroups of 16 segments (9 with four row blocks and four groups of
//     k), 896 x 4864 13 (37); 9728 x 896 10.7 with four row blocks (12), 151936 x 896 98 with eight (113);
//   more: the largest tile that still leaves the 256 compute units evenly loaded.  896 x 896 at 64 / 128 / 509 /
//     1024 rows 5.7 / 7.3 / 17 / 26 (16 x 16, 32 x 16, 32 x 64, 64 x 64), 9728 x 896 at 64 / 509 25 / 124
//     (32 x 32, 64 x 64: 70 TFLOP/s of the 150 that the instruction reaches alone).  A k of up to 256 is one step
//     a segment, and a shorter one leaves the later of four groups without any: there a wavefront walks all of k and
//     four lie side by side along the rows.  1,501 rows: 28 products of 448 x 128 160 us shared by four groups, 77 so
//     (95 with vector instructions), 14 of 128 x 64 27, 13 (14), 40 of 256 x 192 132, 86 (105), 4864 x 256 73, 55 (66).
template <bool TILED>
static void run_f32(const F32Product& p, hipStream_t s) {
  auto tiles = [&](int rows, int cols) {
    return static_cast<long long>((p.m + rows - 1) / rows) * ((p.n + cols - 1) / cols) * p.batch;
  };
  auto one_round = [](long long count) { return count >= 192 && count <= 256; };
  if (p.n <= 16) {
    if (p.m <= 2048)
      launch_f32<1, 1, 16, 1, 1, 2, TILED>(p, s);
    else if (p.m <= 32768)
      launch_f32<1, 1, 4, 4, 1, 4, TILED>(p, s);
    else
      launch_f32<2, 1, 4, 4, 1, 2, TILED>(p, s);
  } else if (tiles(64, 64) >= 640 || one_round(tiles(64, 64))) {
    if (p.k <= 256)
      launch_f32<4, 2, 1, 1, 4, 1, TILED>(p, s);
    else
      launch_f32<4, 4, 4, 1, 1, 1, TILED>(p, s);
  } else if (one_round(tiles(32, 64))) {
    launch_f32<2, 4, 4, 1, 1, 2, TILED>(p, s);
  } else if (tiles(16, 16) <= 256) {
    launch_f32<1, 1, 16, 1, 1, 2, TILED>(p, s);
  } else if (tiles(32, 16) <= 256) {
    launch_f32<2, 1, 16, 1, 1, 2, TILED>(p, s);
  } else {
    launch_f32<2, 2, 4, 1, 1, 2, TILED>(p, s);
  }
}

void gemm_f32(const float* a, const float* w, bool tiled, const float* bias, float* out, int n, int m, int k, int lda,
              int ldo, int accumulate, int batch, long long a_batch, long long w_batch, long long out_batch,
              hipStream_t s) {
  const F32Product p{a, w, bias, out, n, m, k, lda, ldo, accumulate, batch, a_batch, w_batch, out_batch};
  if (tiled)
    run_f32<true>(p, s);
  else
    run_f32<false>(p, s);
}

// wt[m / 16][k / 16][64 lanes][4]: lane 16 g + i of a tile holds elements 4 g .. 4 g + 3 of row i, zeros
// beyond the matrix.
__global__ void __launch_bounds__(256)
    retile_f32_kernel(const float* __restrict__ w, int m, int k, float* __restrict__ wt, long long quads) {
  const long long q = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
  if (q >= quads) return;
  const int ktiles = (k + 15) / 16, lane = q % 64;
  const long long tile = q / 64;
  const long long row = tile / ktiles * 16 + lane % 16;
  const int col = static_cast<int>(tile % ktiles) * 16 + lane / 16 * 4;
  mf4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = row < m && col + e < k ? w[row * k + col + e] : 0.f;
  *reinterpret_cast<mf4*>(wt + q * 4) = v;
}

}  // namespace shk

using namespace shk;

extern "C" int shk_retile_f32(const void* w, int m, int k, void* wt, void* stream) {
  SHK_REQUIRE(m > 0 && k > 0, "retile_f32: bad sizes m=%d k=%d", m, k);
  SHK_REQUIRE(w && wt && reinterpret_cast<uintptr_t>(wt) % 16 == 0, "retile_f32: null or misaligned pointer");
  const long long quads = static_cast<long long>((m + 15) / 16) * ((k + 15) / 16) * 64;
  SHK_REQUIRE((quads + 255) / 256 < (1LL << 31), "retile_f32: the matrix is too large");
  retile_f32_kernel<<<static_cast<unsigned>((quads + 255) / 256), 256, 0, static_cast<hipStream_t>(stream)>>>(
      static_cast<const float*>(w), m, k, static_cast<float*>(wt), quads);
  SHK_LAUNCH_CHECK("retile_f32");
  return 0;
}

extern "C" int shk_gemm_f32_tiled_weight(const void* a, const void* wt, const float* bias, void* out, int n, int m, int k,
                                         int lda, int ldo, int accumulate, void* stream) {
  SHK_REQUIRE(n >= 0 && m > 0 && k > 0, "gemm_f32: bad sizes n=%d m=%d k=%d", n, m, k);
  SHK_REQUIRE(lda >= k && ldo >= m, "gemm_f32: row strides lda=%d ldo=%d too small for k=%d m=%d", lda, ldo, k, m);
  if (n == 0) return 0;
  SHK_REQUIRE(a && wt && out && reinterpret_cast<uintptr_t>(wt) % 16 == 0, "gemm_f32: null or misaligned pointer");
  SHK_REQUIRE((n + 63) / 64 <= 65535, "gemm_f32: too many rows (%d)", n);
  gemm_f32(static_cast<const float*>(a), static_cast<const float*>(wt), true, bias, static_cast<float*>(out), n, m, k, lda,
           ldo, accumulate, 1, 0, 0, 0, static_cast<hipStream_t>(stream));
  SHK_LAUNCH_CHECK("gemm_f32");
  return 0;
}
