// out[n, m] = a[n, k] @ w[m, k]^T + bias: the matrix products of the model
// (projections, feed-forward, output matrix).
//
// gemm_tiled_kernel is the general kernel of bfloat16 operands: every size, float32
// fused-multiply-add accumulation in ascending k for every output element; the
// fallback of the bfloat16 path.  float32 operands go to gemm_f32.hip.
#include "api.h"
#include "common.h"
#include "to_lds.h"

namespace shk {

constexpr int kTM = 64;  // rows of a (tokens) per workgroup
constexpr int kTN = 64;  // rows of w (output features) per workgroup
constexpr int kTK = 16;  // depth of one staged slice

template <typename TI, typename TO>
__global__ void __launch_bounds__(256)
    gemm_tiled_kernel(const TI* __restrict__ a, const TI* __restrict__ w,
                      const float* __restrict__ bias, TO* __restrict__ out, int n, int m, int k,
                      int lda, int ldo, int accumulate, long long a_batch, long long w_batch,
                      long long out_batch) {
  // blockIdx.z: one of a batch of products of equal shape, operands a fixed step apart
  a += blockIdx.z * a_batch;
  w += blockIdx.z * w_batch;
  out += blockIdx.z * out_batch;
  __shared__ float as[kTK][kTM + 4];
  __shared__ float ws[kTK][kTN + 4];
  const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
  const int row0 = blockIdx.y * kTM, col0 = blockIdx.x * kTN;

  float acc[4][4] = {};
  for (int k0 = 0; k0 < k; k0 += kTK) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int idx = threadIdx.x + i * 256;  // 0..1023 over [64 rows][16 k]
      const int r = idx / kTK, kk = idx % kTK;
      const int gr = row0 + r, gc = col0 + r, gk = k0 + kk;
      as[kk][r] = (gr < n && gk < k) ? to_float(a[static_cast<size_t>(gr) * lda + gk]) : 0.f;
      ws[kk][r] = (gc < m && gk < k) ? to_float(w[static_cast<size_t>(gc) * k + gk]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < kTK; ++kk) {
      float av[4], wv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) av[i] = as[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) wv[j] = ws[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(av[i], wv[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int gr = row0 + ty * 4 + i;
    if (gr >= n) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int gc = col0 + tx * 4 + j;
      if (gc >= m) continue;
      float v = acc[i][j];
      if (bias) v += bias[gc];
      TO* dst = out + static_cast<size_t>(gr) * ldo + gc;
      if (accumulate) v += to_float(*dst);
      *dst = from_float<TO>(v);
    }
  }
}

// A batch of products with few rows of a (single tokens): one wavefront per (product of the
// batch, output feature) walks that weight row once, every lane a run of it, and forms the dot
// products of up to 16 rows of a at a time; sums over the lanes in a fixed order.  Weight rows
// are read whole and once, and thousands of wavefronts keep the memory busy, where the tiled
// kernel's few workgroups would each walk a long k alone.
constexpr int kSkinnyRows = 16;

template <typename T, typename TO>
__global__ void __launch_bounds__(256)
    gemm_batched_skinny_kernel(const T* __restrict__ a, const T* __restrict__ w, TO* __restrict__ out, int n,
                               int m, int k, int lda, int ldo, long long a_batch, long long w_batch,
                               long long out_batch) {
  const int lane = threadIdx.x % kWave;
  const int row = blockIdx.x * (256 / kWave) + threadIdx.x / kWave;  // output feature
  if (row >= m) return;
  const int b = blockIdx.y;
  const T* wr = w + b * w_batch + static_cast<size_t>(row) * k;
  const T* ab = a + b * a_batch;
  for (int n0 = 0; n0 < n; n0 += kSkinnyRows) {
    float acc[kSkinnyRows];
#pragma unroll
    for (int r = 0; r < kSkinnyRows; ++r) acc[r] = 0.f;
    for (int kk = lane; kk < k; kk += kWave) {
      const float wv = to_float(wr[kk]);
#pragma unroll
      for (int r = 0; r < kSkinnyRows; ++r)
        if (n0 + r < n) acc[r] = fmaf(to_float(ab[static_cast<size_t>(n0 + r) * lda + kk]), wv, acc[r]);
    }
#pragma unroll
    for (int r = 0; r < kSkinnyRows; ++r) {
      const float total = wave_sum(acc[r]);
      if (lane == 0 && n0 + r < n) out[b * out_batch + static_cast<size_t>(n0 + r) * ldo + row] = from_float<TO>(total);
    }
  }
}

// gemm_f32.hip
void gemm_f32(const float* a, const float* w, bool tiled, const float* bias, float* out, int n, int m, int k, int lda,
              int ldo, int accumulate, int batch, long long a_batch, long long w_batch, long long out_batch,
              hipStream_t s);

template <typename TI, typename TO>
static int launch_tiled(const void* a, const void* w, const float* bias, void* out, int n, int m,
                        int k, int lda, int ldo, int accumulate, hipStream_t s, int batch = 1,
                        long long a_batch = 0, long long w_batch = 0, long long out_batch = 0) {
  dim3 grid((m + kTN - 1) / kTN, (n + kTM - 1) / kTM, batch);
  gemm_tiled_kernel<TI, TO><<<grid, 256, 0, s>>>(static_cast<const TI*>(a),
                                                 static_cast<const TI*>(w), bias,
                                                 static_cast<TO*>(out), n, m, k, lda, ldo,
                                                 accumulate, a_batch, w_batch, out_batch);
  return 0;
}

}  // namespace shk

using namespace shk;

extern "C" int shk_gemm(const void* a, const void* w, const float* bias, void* out, int n, int m,
                        int k, int lda, int ldo, int in_dtype, int out_dtype, int accumulate,
                        void* stream) {
  SHK_REQUIRE(in_dtype == kF32 || in_dtype == kBF16, "gemm: unknown in_dtype %d", in_dtype);
  SHK_REQUIRE(out_dtype == kF32 || out_dtype == kBF16, "gemm: unknown out_dtype %d", out_dtype);
  SHK_REQUIRE(n >= 0 && m > 0 && k > 0, "gemm: bad sizes n=%d m=%d k=%d", n, m, k);
  SHK_REQUIRE(lda >= k && ldo >= m, "gemm: row strides lda=%d ldo=%d too small for k=%d m=%d", lda,
              ldo, k, m);
  SHK_REQUIRE(!accumulate || out_dtype == kF32, "gemm: accumulate needs a float32 output");
  SHK_REQUIRE(!(in_dtype == kF32 && out_dtype == kBF16),
              "gemm: float32 inputs with a bfloat16 output are not built");
  if (n == 0) return 0;
  SHK_REQUIRE(a && w && out, "gemm: null pointer");
  SHK_REQUIRE((n + kTM - 1) / kTM <= 65535, "gemm: too many rows (%d)", n);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (in_dtype == kF32)
    gemm_f32(static_cast<const float*>(a), static_cast<const float*>(w), false, bias, static_cast<float*>(out), n, m, k, lda,
             ldo, accumulate, 1, 0, 0, 0, s);
  else if (out_dtype == kF32)
    launch_tiled<bf16, float>(a, w, bias, out, n, m, k, lda, ldo, accumulate, s);
  else
    launch_tiled<bf16, bf16>(a, w, bias, out, n, m, k, lda, ldo, accumulate, s);
  SHK_LAUNCH_CHECK("gemm");
  return 0;
}

// The same batch on the matrix units for bfloat16: both operands are row-major with k innermost, which
// is the operand layout of v_mfma_f32_16x16x32_bf16 as it stands (a lane's 8 consecutive k of one row
// are one 16-byte load), so nothing passes through LDS.  A wavefront forms RT x CT tiles of 16 rows x
// 16 features, a workgroup RW x CW of that; the next U steps' operands are in flight while U are
// multiplied.  k in multiples of 8 and 16-byte aligned rows; sums run over k in ascending order in every
// shape, so a row's result depends neither on the shape nor on what else is in the step.
// What bounds it is the compute units' intake: 64 x 64 a wavefront needs 8 KiB for 16 instructions.
// 28 heads, 1,501 rows (which the next kernel takes now): k = 128 to 448 features 74 us with 16 x 64 a wavefront, no load ahead and 2-byte
// stores, 41 so; k = 448 to 128 features 58, now 35; 14 blocks of 256 to 512 float32 68, now 35.  Eight rows: 6.0,
// 11.7 and 7.5 us with 64-row workgroups, 5.0, 5.9 and 4.7 now.
typedef __bf16 gbf16x8 __attribute__((ext_vector_type(8)));
typedef float gf32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int gu32x4 __attribute__((ext_vector_type(4)));

template <int RT, int CT, int RW, int CW, int U, typename TO>
__global__ void __launch_bounds__(kWave* RW* CW)
    gemm_batched_mfma_kernel(const bf16* __restrict__ a, const bf16* __restrict__ w, TO* __restrict__ out, int n,
                             int m, int k, int lda, int ldo, int vec_out, long long a_batch, long long w_batch,
                             long long out_batch) {
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int i = lane % 16, kg = lane / 16;
  const int b = blockIdx.z;
  const int row0 = (blockIdx.y * RW + wave / CW) * RT * 16, col0 = (blockIdx.x * CW + wave % CW) * CT * 16;
  if (row0 >= n || col0 >= m) return;  // (no barrier in this kernel)
  // rows beyond either matrix are read as its last and not stored
  const bf16 *ar[RT], *wr[CT];
#pragma unroll
  for (int r = 0; r < RT; ++r) ar[r] = a + b * a_batch + static_cast<size_t>(min(row0 + r * 16 + i, n - 1)) * lda + kg * 8;
#pragma unroll
  for (int c = 0; c < CT; ++c) wr[c] = w + b * w_batch + static_cast<size_t>(min(col0 + c * 16 + i, m - 1)) * k + kg * 8;
  gf32x4 acc[RT][CT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[r][c] = gf32x4{0.f, 0.f, 0.f, 0.f};
  // the products are formed transposed (features as rows): a lane gets features 4 kg + 0..3 of a tile for row i
  auto multiply = [&](const gu32x4(&av)[RT], const gu32x4(&wv)[CT]) {
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int c = 0; c < CT; ++c)
        acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gbf16x8, wv[c]),
                                                            __builtin_bit_cast(gbf16x8, av[r]), acc[r][c], 0, 0, 0);
  };
  const int steps = k / 32;
  if (steps > 0) {
    gu32x4 av[2][U][RT], wv[2][U][CT];
    auto load = [&](int set, int s0) {
#pragma unroll
      for (int u = 0; u < U; ++u) {  // (unconditional: a step beyond the last is the last again)
        const int kk = min(s0 + u, steps - 1) * 32;
#pragma unroll
        for (int r = 0; r < RT; ++r) av[set][u][r] = *reinterpret_cast<const gu32x4*>(ar[r] + kk);
#pragma unroll
        for (int c = 0; c < CT; ++c) wv[set][u][c] = *reinterpret_cast<const gu32x4*>(wr[c] + kk);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    load(0, 0);
    for (int s = 0; s < steps; s += 2 * U) {
      load(1, s + U);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (s + u < steps) multiply(av[0][u], wv[0][u]);
      load(0, s + 2 * U);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (s + U + u < steps) multiply(av[1][u], wv[1][u]);
    }
  }
  if (steps * 32 < k) {  // (k is a multiple of 8: a lane's piece is whole or absent)
    const bool have = steps * 32 + kg * 8 < k;
    const int kk = have ? steps * 32 : -kg * 8;
    const uint32_t keep = have ? 0xffffffffu : 0u;
    gu32x4 av[RT], wv[CT];
#pragma unroll
    for (int r = 0; r < RT; ++r) av[r] = *reinterpret_cast<const gu32x4*>(ar[r] + kk) & keep;
#pragma unroll
    for (int c = 0; c < CT; ++c) wv[c] = *reinterpret_cast<const gu32x4*>(wr[c] + kk) & keep;
    multiply(av, wv);
  }
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int row = row0 + r * 16 + i;
    if (row >= n) continue;
    TO* dst = out + b * out_batch + static_cast<size_t>(row) * ldo;
#pragma unroll
    for (int t = 0; t < CT; ++t) {
      const int c = col0 + t * 16 + 4 * kg;
      if (vec_out && c + 3 < m) {
        if constexpr (sizeof(TO) == 4) {
          *reinterpret_cast<gf32x4*>(dst + c) = acc[r][t];
        } else {
          const uint32_t lo = bf16_bits(acc[r][t][0]) | static_cast<uint32_t>(bf16_bits(acc[r][t][1])) << 16;
          const uint32_t hi = bf16_bits(acc[r][t][2]) | static_cast<uint32_t>(bf16_bits(acc[r][t][3])) << 16;
          *reinterpret_cast<uint2*>(dst + c) = make_uint2(lo, hi);
        }
        continue;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c + e < m) dst[c + e] = from_float<TO>(acc[r][t][e]);
    }
  }
}

// The same for many rows and k in whole stages of 64: both operands go straight into LDS in whole cache lines, 8 rows x 128 bytes a
// load (a compute unit takes in loads of 16 rows x 64 bytes at a quarter of its rate, and a workgroup's four wavefronts asked for
// everything twice), and results leave through LDS in whole pieces along the rows.  128 rows x 128 features a workgroup, two
// of which share a compute unit; two stages in LDS, one in flight while the other is multiplied.  The same instructions in the
// same order of k: the same bits.  28 heads, 1,501 rows, in prompts: k = 128 to 448 features 42.4 us in the kernel above, 26.8 so, k = 448 to
// 128 features 36.3, 17.3; 14 blocks of 256 to 512 float32 35.7, 19.9.  What bounds it now: a workgroup's chain of two to seven stages' latency and four
// turns of its results through LDS, which only one other workgroup on the compute unit covers; the results alone, 38 to 43 MB but for the second, would
// take a third to a half of that at a copy's rate.
constexpr int kLinesK = 64, kLinesRows = 128;

template <typename TO>
__global__ void __launch_bounds__(4 * kWave)
    gemm_batched_lines_kernel(const bf16* __restrict__ a, const bf16* __restrict__ w, TO* __restrict__ out, int n, int m, int k,
                              int lda, int ldo, long long a_batch, long long w_batch, long long out_batch) {
  constexpr int kUnits = kLinesRows / 8, kLoads = 2 * kUnits / 4;  // units of 8 rows of an operand's stage; a wavefront's loads of a stage
  __shared__ gu32x4 mem[2 * 2 * kUnits * kWave];                    // stages, each rows then features
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int i = lane % 16, kg = lane / 16;
  const int row0 = blockIdx.y * kLinesRows, col0 = blockIdx.x * kLinesRows, stages = k / kLinesK;
  const char* asrc = reinterpret_cast<const char*>(a + blockIdx.z * a_batch + static_cast<size_t>(row0) * lda);
  const char* wsrc = reinterpret_cast<const char*>(w + blockIdx.z * w_batch + static_cast<size_t>(col0) * k);
  const unsigned base = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)mem));
  // Lane l of a unit loads piece (l % 8) ^ (l / 8) of row l / 8: reads of 16 rows at one piece then meet no bank conflicts.
  // Rows beyond either matrix are read as its last and not stored.
  unsigned aoff[kLoads / 2], woff[kLoads / 2];
#pragma unroll
  for (int u = 0; u < kLoads / 2; ++u) {
    const int row = (wave + 4 * u) * 8 + lane / 8;
    const unsigned piece = ((lane % 8) ^ (lane / 8)) * 16u;
    aoff[u] = static_cast<unsigned>(min(row, n - 1 - row0)) * lda * 2u + piece;
    woff[u] = static_cast<unsigned>(min(row, m - 1 - col0)) * k * 2u + piece;
  }
  auto load = [&](int st) {  // (a stage beyond the last: the last again, never multiplied)
    const size_t at = static_cast<size_t>(min(st, stages - 1)) * (kLinesK * 2);
    const unsigned to = base + (st % 2 * 2 * kUnits + wave) * 1024;
#pragma unroll
    for (int u = 0; u < kLoads / 2; ++u) SHK_LOAD_TO_LDS(to + u * 4096, aoff[u], asrc + at);
#pragma unroll
    for (int u = 0; u < kLoads / 2; ++u) SHK_LOAD_TO_LDS(to + kUnits * 1024 + u * 4096, woff[u], wsrc + at);
  };
  gf32x4 acc[4][4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[r][c] = gf32x4{0.f, 0.f, 0.f, 0.f};
  const int arow = wave / 2 * 64, wrow = wave % 2 * 64;
  load(0);
  load(1);
  for (int st = 0; st < stages; ++st) {
    SHK_MEET_WITH_LOADS(kLoads);  // (the stage has landed for every wavefront)
    const char* lds = reinterpret_cast<const char*>(mem) + st % 2 * 2 * kUnits * 1024;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int piece = ((4 * h + kg) ^ (i % 8)) * 16;
      gu32x4 av[4], wv[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) av[r] = *reinterpret_cast<const gu32x4*>(lds + (arow + r * 16 + i) * 128 + piece);
#pragma unroll
      for (int c = 0; c < 4; ++c) wv[c] = *reinterpret_cast<const gu32x4*>(lds + (kLinesRows + wrow + c * 16 + i) * 128 + piece);
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gbf16x8, wv[c]), __builtin_bit_cast(gbf16x8, av[r]),
                                                              acc[r][c], 0, 0, 0);
    }
    SHK_MEET_WITH_LOADS(kLoads);  // (nobody reads the stage any more; only the next one's loads are in flight)
    load(st + 2);
  }
  SHK_WAIT_LOADS(0);
  __syncthreads();
  // A lane has features 4 kg + 0..3 of a tile for row i.  Sixteen rows of a wavefront at a time, in two places by turns.
  constexpr int E = sizeof(TO), kPitch = 64 * E + 16, kPieces = 64 * E / 16;
  static_assert(4 * 2 * 16 * kPitch <= sizeof(mem), "the results of sixteen rows a wavefront fit LDS twice");
  char* mine = reinterpret_cast<char*>(mem) + wave * 2 * 16 * kPitch;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    char* place = mine + r % 2 * 16 * kPitch;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      char* to = place + i * kPitch + (t * 16 + 4 * kg) * E;
      if constexpr (E == 4) {
        *reinterpret_cast<gf32x4*>(to) = acc[r][t];
      } else {
        const uint32_t lo = bf16_bits(acc[r][t][0]) | static_cast<uint32_t>(bf16_bits(acc[r][t][1])) << 16;
        const uint32_t hi = bf16_bits(acc[r][t][2]) | static_cast<uint32_t>(bf16_bits(acc[r][t][3])) << 16;
        *reinterpret_cast<uint2*>(to) = make_uint2(lo, hi);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int q = 0; q < 16 * kPieces / kWave; ++q) {
      const int t = (q * kWave + lane) / kPieces, p = (q * kWave + lane) % kPieces;
      const int row = row0 + arow + r * 16 + t, col = col0 + wrow + p * (16 / E);
      const gu32x4 v = *reinterpret_cast<const gu32x4*>(place + t * kPitch + p * 16);
      if (row < n && col < m) *reinterpret_cast<gu32x4*>(out + blockIdx.z * out_batch + static_cast<size_t>(row) * ldo + col) = v;
    }
  }
}

// The fewest rows of whole lines and pieces for which gemm_batched_lines_kernel is the faster one, where its workgroups fill the compute units: each
// loads 128 rows and forms 128 features, however few there are, and rounds them all where the results are bfloat16.  Weights cold, us at 1 / 8 / 16 /
// 17 / 48 / 64 rows in the other kernels and in this one:
//   256 of k = 64 to 128 features   bfloat16 3.7 / 4.0 / 4.5 / 5.7 / 7.1 / 8.2 and 5.8 / 5.9 / 6.1 / 6.1 / 6.9 / 7.3,
//                                   float32 3.6 / 4.1 / 4.7 / 4.9 / 6.5 / 7.2 and 4.1 / 4.3 / 4.7 / 4.9 / 6.0 / 6.6
//   128 of 128 to 256               bfloat16 6.0 / 7.1 / 8.1 / 7.5 / 9.0 / 10.1 and 6.9 / 7.0 / 7.1 / 7.1 / 7.8 / 8.3,
//                                   float32 6.1 / 7.1 / 8.3 / 6.6 / 8.2 / 9.0 and 5.3 / 5.5 / 5.7 / 5.8 / 6.9 / 7.7
//   256 of 192 to 128               bfloat16 6.2 / 7.3 / 8.6 / 9.2 / 10.9 / 12.3 and 7.6 / 7.9 / 8.1 / 8.2 / 9.1 / 9.7
//   128 of 512 to 256               bfloat16 10.1 / 11.3 / 13.1 / 16.9 / 19.1 / 20.8 and 12.9 / 12.9 / 12.9 / 13.0 / 14.3 / 15.1
// With up to 64 features half of it is idle: 256 of 128 to 64 a quarter to a half slower up to 16 rows, 7 % at 17 to 32, 14 % faster from 49 on.
static int batched_lines_from(int m, int k, bool f32) {
  if (k < 128 || (m <= 64 && k < 192)) return 49;
  if (m <= 64) return 17;
  return f32 && k < 256 ? 1 : (k < 256 ? k : 256) / 16 + 1;
}

static bool batched_lines(int n, int m, int k, int batch, bool f32) {
  const long long groups = static_cast<long long>((m + kLinesRows - 1) / kLinesRows) * ((n + kLinesRows - 1) / kLinesRows) * batch;
  return k % kLinesK == 0 && k <= 1 << 22 && groups >= 256 && n >= batched_lines_from(m, k, f32);
}

// Shapes: up to 16 rows 16 x 16 a wavefront, side by side along the features (the weights' latency is all
// there is); 64 x 64 a wavefront where such workgroups fill the compute units, else 32 x 32; through LDS where batched_lines() says so and k and
// the results are whole lines and pieces.  A k of one or two steps
// is loaded a step at a time: eight steps' loads, most of them the last step's again, took 4.1 us for 8 products
// of 256 x 64 at 16 rows, two 2.4 (3.1 with 64-row workgroups).
template <typename TO>
static void launch_batched_mfma(const bf16* a, const bf16* w, TO* out, int n, int m, int k, int lda, int ldo, int batch,
                                long long a_batch, long long w_batch, long long out_batch, hipStream_t s) {
  const int vec_out = ldo % 4 == 0 && out_batch % 4 == 0 && reinterpret_cast<uintptr_t>(out) % (4 * sizeof(TO)) == 0;
  auto grid = [&](int rows, int cols) { return dim3((m + cols - 1) / cols, (n + rows - 1) / rows, batch); };
  const dim3 large = grid(128, 128);
  const bool short_k = k <= 64;
  const int per = 16 / sizeof(TO);  // values of a piece
  // whole stages and whole pieces everywhere, offsets within a workgroup's rows in 32 bits
  const bool whole = m % per == 0 && ldo % per == 0 && out_batch % per == 0 && w_batch % 8 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0 && lda <= 1 << 22;
  if (whole && batched_lines(n, m, k, batch, sizeof(TO) == 4))
    gemm_batched_lines_kernel<TO><<<large, 256, 0, s>>>(a, w, out, n, m, k, lda, ldo, a_batch, w_batch, out_batch);
  else if (n <= 16 && short_k)
    gemm_batched_mfma_kernel<1, 1, 1, 4, 1, TO>
        <<<grid(16, 64), 256, 0, s>>>(a, w, out, n, m, k, lda, ldo, vec_out, a_batch, w_batch, out_batch);
  else if (n <= 16)
    gemm_batched_mfma_kernel<1, 1, 1, 4, 4, TO>
        <<<grid(16, 64), 256, 0, s>>>(a, w, out, n, m, k, lda, ldo, vec_out, a_batch, w_batch, out_batch);
  else if (static_cast<long long>(large.x) * large.y * batch >= 256)
    gemm_batched_mfma_kernel<4, 4, 2, 2, 1, TO>
        <<<large, 256, 0, s>>>(a, w, out, n, m, k, lda, ldo, vec_out, a_batch, w_batch, out_batch);
  else if (short_k)
    gemm_batched_mfma_kernel<2, 2, 2, 2, 1, TO>
        <<<grid(64, 64), 256, 0, s>>>(a, w, out, n, m, k, lda, ldo, vec_out, a_batch, w_batch, out_batch);
  else
    gemm_batched_mfma_kernel<2, 2, 2, 2, 2, TO>
        <<<grid(64, 64), 256, 0, s>>>(a, w, out, n, m, k, lda, ldo, vec_out, a_batch, w_batch, out_batch);
}

// Whether bfloat16 operands in whole lines whose results are whole pieces (`f32`: of float32) go through LDS.
extern "C" int shk_gemm_batched_lines(int n, int m, int k, int batch, int f32) {
  return n > 0 && m > 0 && k > 0 && batch > 0 && batched_lines(n, m, k, batch, f32);
}

// A batch of products of one shape (one per head, say): product b reads a + b * a_batch
// (rows lda apart), w + b * w_batch ([m, k] contiguous) and writes out + b * out_batch.
extern "C" int shk_gemm_batched(const void* a, const void* w, void* out, int n, int m, int k, int lda,
                                int ldo, int batch, long long a_batch, long long w_batch,
                                long long out_batch, int dtype, int out_dtype, void* stream) {
  SHK_REQUIRE(dtype == kF32 || dtype == kBF16, "gemm_batched: unknown dtype %d", dtype);
  SHK_REQUIRE(out_dtype == dtype || out_dtype == kF32, "gemm_batched: outputs are of the operands' dtype or float32");
  SHK_REQUIRE(n >= 0 && m > 0 && k > 0 && batch > 0 && batch <= 65535, "gemm_batched: bad sizes n=%d m=%d k=%d batch=%d",
              n, m, k, batch);
  SHK_REQUIRE(lda >= k && ldo >= m, "gemm_batched: row strides lda=%d ldo=%d too small for k=%d m=%d", lda, ldo, k, m);
  SHK_REQUIRE(a_batch >= 0 && w_batch >= 0 && out_batch >= m, "gemm_batched: outputs of the batch would overlap");
  if (n == 0) return 0;
  SHK_REQUIRE(a && w && out, "gemm_batched: null pointer");
  SHK_REQUIRE((n + kTM - 1) / kTM <= 65535, "gemm_batched: too many rows (%d)", n);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == kBF16 && k % 8 == 0 && lda % 8 == 0 && a_batch % 8 == 0 && reinterpret_cast<uintptr_t>(a) % 16 == 0 &&
      reinterpret_cast<uintptr_t>(w) % 16 == 0 && (n + 63) / 64 <= 65535) {
    const bf16 *ab = static_cast<const bf16*>(a), *wb = static_cast<const bf16*>(w);
    if (out_dtype == kF32)
      launch_batched_mfma(ab, wb, static_cast<float*>(out), n, m, k, lda, ldo, batch, a_batch, w_batch, out_batch, s);
    else
      launch_batched_mfma(ab, wb, static_cast<bf16*>(out), n, m, k, lda, ldo, batch, a_batch, w_batch, out_batch, s);
  } else if (n <= 2 * kSkinnyRows && dtype == kBF16) {
    // (float32 keeps one order of summation whatever the number of rows: gemm_f32.hip)
    dim3 grid((m + 3) / 4, batch);
    if (out_dtype == kF32)
      gemm_batched_skinny_kernel<bf16, float><<<grid, 256, 0, s>>>(static_cast<const bf16*>(a), static_cast<const bf16*>(w),
                                                                   static_cast<float*>(out), n, m, k, lda, ldo, a_batch,
                                                                   w_batch, out_batch);
    else
      gemm_batched_skinny_kernel<bf16, bf16><<<grid, 256, 0, s>>>(static_cast<const bf16*>(a), static_cast<const bf16*>(w),
                                                                  static_cast<bf16*>(out), n, m, k, lda, ldo, a_batch,
                                                                  w_batch, out_batch);
  } else if (dtype == kF32)
    gemm_f32(static_cast<const float*>(a), static_cast<const float*>(w), false, nullptr, static_cast<float*>(out), n, m, k,
             lda, ldo, 0, batch, a_batch, w_batch, out_batch, s);
  else if (out_dtype == kF32)
    launch_tiled<bf16, float>(a, w, nullptr, out, n, m, k, lda, ldo, 0, s, batch, a_batch, w_batch, out_batch);
  else
    launch_tiled<bf16, bf16>(a, w, nullptr, out, n, m, k, lda, ldo, 0, s, batch, a_batch, w_batch, out_batch);
  SHK_LAUNCH_CHECK("gemm_batched");
  return 0;
}
