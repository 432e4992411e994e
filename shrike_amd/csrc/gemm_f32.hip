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
// many the supply of operands: a workgroup's wavefronts walk different parts of k and so share no operand (9728 x 896 at 509
// rows 75 TFLOP/s; gemm_f32_lds_kernel, which shares them, 97).  Before, one workgroup per 64 x 64 results with vector
// instructions: a 0.5B decode step of four requests 23.9 ms (2.4 with this kernel, 1.56 with attention_f32.hip as
// well), a 509-token prompt 42.6 ms (18.9, 6.5; 5.4 with operands shared); the logits' error against 64 bits 6.4e-7 (2.5e-7).
#include "api.h"
#include "common.h"
#include "gemm_wide.h"

#include <type_traits>

namespace shk {

typedef float mf4 __attribute__((ext_vector_type(4)));

constexpr int kF32Segments = 16, kF32Group = 4;

// act(gate) * up as act_mul_kernel forms it
struct F32Gate {
  int act;
  float limit, up_shift;
};
__device__ __forceinline__ float f32_gate(float g, float u, F32Gate gate) {
  if (gate.limit > 0.f) {
    g = fminf(g, gate.limit);
    u = fminf(fmaxf(u, -gate.limit), gate.limit);
  }
  u += gate.up_shift;
  if (gate.act == 3) return fmaxf(g, 0.f) * u;
  const float x = gate.act == 2 ? 2.f * 0.7978845608028654f * (g + 0.044715f * g * g * g) : gate.act == 4 ? 1.702f * g : g;
  return g / (1.f + expf(-x)) * u;
}
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

// The same product, in the same order, for up to 16 rows, tiled weights and a k in whole steps of 16.  A workgroup's KW
// wavefronts take a segment each (16), a group each (4), or with GROUPS the segments of the group blockIdx.y, whose sum is then
// one of four parts [group][n][m] that the reader adds in order.  C > 0: a wavefront has at most C steps, all asked for at
// once; 0: batches of five, two in flight.  ROWS = 8: a workgroup for half a block of features, where whole blocks leave
// compute units idle.  GATED: w holds a gate matrix and behind it the other factor, m rows each (a multiple of 16); a workgroup
// forms a block of both and stores what act_mul_kernel would of the two.
// What bounds it: one round trip to memory, then the matrix instructions (32 cycles each, 16 columns for however few rows).  Weights cold, us at 1 /
// 4 / 16 rows: 896 x 896 4.8 / 5.0 / 6.4 in the kernel above, 3.8 / 3.9 / 4.5 here, 9728 x 896 11.1 / 10.5 / 13.0 and 8.8 / 8.9 / 10.2,
// 3584 x 3584 28 / 29 / 39 and 12 / 12 / 15.
// A wavefront's part of the rows is loaded in whole lines and handed to the lanes that multiply it through LDS, in a place of the wavefront's own:
// straight from memory neighbouring lanes lie on different rows, which a compute unit takes in at a quarter of its rate.  At 4 / 8 / 16 rows: 1152 x 896
// 4.1 / 4.4 / 5.1 -> 4.0 / 4.1 / 4.5, gate and up of 4864 x 896 10.2 / 10.8 / 12.5 -> 10.0 / 10.3 / 11.4, 896 x 4864 in groups 7.7 / 8.1 / 10.4 -> 7.1 / 7.6 /
// 9.1.  Not where a wavefront walks a group in batches (C = 0, whole): 3584 x 18944 at 4 / 9 50.5 / 51.5 -> 52.0 / 59.2.
// NR: rows that a wavefront holds in LDS (at least n), 0: none.
template <int KW, int ROWS, int C, bool GATED, bool GROUPS, int NR>
struct F32Few {
  static constexpr int kBlocks = GATED ? 2 : 1, kSteps = C > 0 ? C : 5, kParts = kSteps > 6 ? 2 : 1, kHeld = kSteps / kParts;
  static constexpr int kPieces = 4 * kHeld, kPitch = kPieces + 1;  // 16 bytes each: of a row in the steps held at a time; with a place beside them
  static constexpr int kRegion = NR * kPitch > kBlocks * kWave ? NR * kPitch : kBlocks * kWave;  // of a wavefront: its rows, then its sums
  static constexpr int kLds = KW * kRegion * 16;
  static_assert(kLds <= 160 * 1024 && kHeld * kParts == kSteps);
};
template <int KW, int ROWS, int C, bool GATED, bool GROUPS, int NR>
__global__ void __launch_bounds__(kWave* KW)
    gemm_f32_few_kernel(const float* __restrict__ a, const float* __restrict__ w, const float* __restrict__ bias,
                        float* __restrict__ out, int n, int m, int k, int lda, int ldo, int accumulate, F32Gate gate) {
  using F = F32Few<KW, ROWS, C, GATED, GROUPS, NR>;
  constexpr int RB = F::kBlocks, kMine = GROUPS ? 1 : kF32Segments / KW, kSteps = F::kSteps, kHeld = F::kHeld;
  constexpr int kLoads = NR ? (NR * F::kPieces + kWave - 1) / kWave : kHeld;  // of a wavefront's rows, for the steps held at a time
  static_assert(!GROUPS || (KW == kF32Group && !GATED), "a workgroup holds one group");
  extern __shared__ mf4 mem[];  // [KW][kRegion]
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int i = lane % 16, kg = lane / 16;
  const int f = blockIdx.x * ROWS + i % ROWS, ktiles = k / 16;
  const mf4* wr[RB];
#pragma unroll
  for (int r = 0; r < RB; ++r)
    wr[r] = reinterpret_cast<const mf4*>(w) + static_cast<size_t>(f / 16 + r * (m / 16)) * ktiles * kWave + kg * 16 + f % 16;
  // the rows' pieces that this lane loads, for whichever lane multiplies them
  mf4* held = mem + wave * F::kRegion;
  const float* ar[kLoads];
  int ahead[kLoads], place[kLoads];
#pragma unroll
  for (int t = 0; t < kLoads; ++t) {
    const int at = min(lane + t * kWave, NR * F::kPieces - 1), row = NR ? at / F::kPieces : i, piece = NR ? at % F::kPieces : 4 * t + kg;
    ar[t] = a + static_cast<size_t>(min(row, n - 1)) * lda + piece % 4 * 4;
    ahead[t] = piece / 4, place[t] = row * F::kPitch + piece;
  }
  const mf4* mine = held + (NR ? min(i, min(n, NR) - 1) * F::kPitch + kg : 0);

  const int seg_steps = (k + 16 * kF32Segments - 1) / (16 * kF32Segments);
  const int first = (GROUPS ? blockIdx.y * kF32Group : 0) + wave * kMine;
  const int begin = min(first * seg_steps, ktiles), steps = min(begin + kMine * seg_steps, ktiles) - begin;
  mf4 acc[RB], group[RB];
#pragma unroll
  for (int r = 0; r < RB; ++r) acc[r] = group[r] = mf4{0.f, 0.f, 0.f, 0.f};
  struct Batch {
    mf4 w[kSteps][RB], a[F::kParts][kLoads];
  };
  auto load = [&](Batch& b, int s0) {  // (unconditional: a step beyond the last is the matrix's last)
#pragma unroll
    for (int part = 0; part < F::kParts; ++part)
#pragma unroll
      for (int t = 0; t < kLoads; ++t)
        b.a[part][t] = *reinterpret_cast<const mf4*>(ar[t] + min(begin + s0 + part * kHeld + ahead[t], ktiles - 1) * 16);
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
      const int s = min(begin + s0 + u, ktiles - 1);
#pragma unroll
      for (int r = 0; r < RB; ++r) b.w[u][r] = __builtin_nontemporal_load(wr[r] + static_cast<size_t>(s) * kWave);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  int in_seg = 0;
  auto multiply = [&](const Batch& b, int s0) {
#pragma unroll
    for (int part = 0; part < F::kParts; ++part) {
      mf4 av[kHeld];
      if constexpr (NR > 0) {
        // (the wavefront's own place: its lanes' writes and reads are in order)
#pragma unroll
        for (int t = 0; t < kLoads; ++t) held[place[t]] = b.a[part][t];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int u = 0; u < kHeld; ++u) av[u] = mine[u * 4];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
      } else {
#pragma unroll
        for (int u = 0; u < kHeld; ++u) av[u] = b.a[part][u];
      }
#pragma unroll
      for (int x = 0; x < kHeld; ++x) {
        const int u = part * kHeld + x;
        // (beyond the last step: zeros times zeros, which leave a sum that began at zero as it is; a branch would take
        // the loads with it)
        const bool have = s0 + u < steps;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float v = have ? av[x][j] : 0.f;
#pragma unroll
          for (int r = 0; r < RB; ++r) acc[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(have ? b.w[u][r][j] : 0.f, v, acc[r], 0, 0, 0);
        }
        if (kMine > 1 && ++in_seg == seg_steps) {  // a segment ends
          in_seg = 0;
#pragma unroll
          for (int r = 0; r < RB; ++r) group[r] += acc[r], acc[r] = mf4{0.f, 0.f, 0.f, 0.f};
        }
      }
    }
  };
  Batch ping;
  load(ping, 0);
  if constexpr (C > 0) {
    multiply(ping, 0);
  } else {
    Batch pong;
    for (int s = 0; s < steps; s += 2 * kSteps) {
      load(pong, s + kSteps);
      multiply(ping, s);
      load(ping, s + 2 * kSteps);
      multiply(pong, s + kSteps);
    }
  }
#pragma unroll
  for (int r = 0; r < RB; ++r) held[r * kWave + lane] = kMine > 1 ? group[r] + acc[r] : acc[r];
  __syncthreads();
  // element (feature, row): the wavefronts' shares in order
  const int row = threadIdx.x / ROWS, at = threadIdx.x % ROWS, col = blockIdx.x * ROWS + at;
  if (row >= n || col >= m) return;
  float v[RB];
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    const float* p = reinterpret_cast<const float*>(mem + r * kWave + at / 4 * 16 + row) + at % 4;
    constexpr int kNext = F::kRegion * 4;
    v[r] = 0.f;
    if (KW > 4) {
#pragma unroll
      for (int g = 0; g < KW; g += KW / 4) {
        float s = 0.f;
#pragma unroll
        for (int x = 0; x < KW / 4; ++x) s += p[(g + x) * kNext];
        v[r] += s;
      }
    } else {
#pragma unroll
      for (int x = 0; x < KW; ++x) v[r] += p[x * kNext];
    }
  }
  float* dst = out + (GROUPS ? static_cast<size_t>(blockIdx.y) * n + row : static_cast<size_t>(row)) * ldo + col;
  if constexpr (GATED) {
    *dst = f32_gate(v[0], v[1], gate);
  } else {
    if (bias) v[0] += bias[col];
    *dst = accumulate ? v[0] + *dst : v[0];
  }
}

template <int KW, int ROWS, int C, bool GATED, bool GROUPS>
static void run_f32_few(const F32Product& p, hipStream_t s, F32Gate gate = F32Gate{}) {
  const auto go = [&](auto kernel, int lds) {
    if (lds > 65536) hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    kernel<<<dim3((p.m + ROWS - 1) / ROWS, GROUPS ? kF32Segments / kF32Group : 1), KW * kWave, lds, s>>>(p.a, p.w, p.bias, p.out, p.n, p.m, p.k, p.lda, p.ldo,
                                                                                                        p.accumulate, gate);
  };
  const auto rows = [&](auto r) {
    using F = F32Few<KW, ROWS, C, GATED, GROUPS, r.value>;
    go(gemm_f32_few_kernel<KW, ROWS, C, GATED, GROUPS, r.value>, F::kLds);
  };
  if constexpr (C == 0 && !GROUPS) {
    rows(std::integral_constant<int, 0>{});
  } else {
    if (p.n <= 4) rows(std::integral_constant<int, 4>{});
    else if (p.n <= 8) rows(std::integral_constant<int, 8>{});
    else if (p.n <= 12) rows(std::integral_constant<int, 12>{});
    else rows(std::integral_constant<int, 16>{});
  }
}

// The same product, in the same order, for many rows and more than 256 of k in whole stages of 32: four wavefronts, 2 x 2 of
// RT x CT tiles, share their operands through LDS, loaded straight into it two stages ahead.  A wavefront walks all of
// k, the tiles' sums of segment, group and all in its registers.  The operands of an instruction's 32 cycles are then a
// quarter of what they are where every wavefront walks a part of k of its own and none shares with another.
// Eight lanes load a row's 128 bytes of a stage, piece c at place c ^ (row / 2 % 8): the 16 lanes that read one piece of 16
// rows meet no bank conflicts.
// What bounds it: the matrix units where workgroups fill the chip several times (3584 x 3584 at 1,501 rows 119 TFLOP/s of
// the 150 that the instruction reaches alone, 9728 x 896 at 509 97).  64 x 64, 128 x 64 and 128 x 128 results a workgroup
// were 4 % slower to twice as slow: fewer wavefronts to cover each other's barriers.  In groups 896 x 4864 at 509 rows, with the norm
// that adds them, 48.6 us, 56.4 whole in gemm_f32_kernel; the gate's two kernels become one, 4864 x 896 at 509 88.1 and 83.2.
// GROUPS: a workgroup forms group blockIdx.y of the sum alone and leaves it in out[blockIdx.y].  GATED: its two blocks of features
// are the gate's and the other factor's, `m` features each.
template <int RT, int CT, bool GATED, bool GROUPS>
__global__ void __launch_bounds__(4 * kWave)
    gemm_f32_lds_kernel(const float* __restrict__ a, const float* __restrict__ w, const float* __restrict__ bias,
                        float* __restrict__ out, int n, int m, int k, int lda, int ldo, int accumulate, int vec_out, F32Gate gate) {
  static_assert(!GATED || (RT == 1 && !GROUPS), "a block of the gate, a block of the other factor");
  constexpr int kRing = 3, kW = 4 * RT, kA = 4 * CT;  // stages; KiB of a stage's weights and rows
  __shared__ mf4 mem[kRing * (kW + kA)][kWave];
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int mw = wave / 2, nw = wave % 2, i = lane % 16, kg = lane / 16;
  // workgroup -> tile as in gemm_f32_kernel
  constexpr int kBlocks = GATED ? 1 : 2 * RT;  // of 16 results a row
  const int rows = (n + 32 * CT - 1) / (32 * CT), cols = (m + 16 * kBlocks - 1) / (16 * kBlocks);
  const int per_die = (rows * cols + kDies - 1) / kDies;
  const int tile = blockIdx.x % kDies * per_die + blockIdx.x / kDies;
  if (blockIdx.x / kDies >= per_die || tile >= rows * cols) return;
  const int f0 = tile / rows * kBlocks, t0 = tile % rows * 32 * CT;  // first block of 16 features, first row
  const int seg_steps = (k + 16 * kF32Segments - 1) / (16 * kF32Segments);
  const int ktiles = k / 16, blocks = (m + 15) / 16;
  // (a group is a whole number of stages; no group of what comes in groups is empty)
  const int first = GROUPS ? blockIdx.y * (kF32Group / 2) * seg_steps : 0;
  const int stages = GROUPS ? min(k / 32 - first, kF32Group / 2 * seg_steps) : k / 32;

  // what a wavefront loads: units wave, wave + 4, ..; rows beyond the last are read as the last and not stored
  unsigned woff[RT], aoff[CT];
#pragma unroll
  for (int u = 0; u < RT; ++u) {
    const int unit = wave + 4 * u, block = GATED ? unit / 2 * blocks : min(f0 + unit / 2, blocks - 1) - f0;
    woff[u] = (static_cast<unsigned>(block) * ktiles + unit % 2) * 1024u + lane * 16u;
  }
#pragma unroll
  for (int u = 0; u < CT; ++u)
    aoff[u] = static_cast<unsigned>(min(t0 + (wave + 4 * u) * 8 + lane / 8, n - 1) - t0) * lda * 4u + ((lane % 8) ^ (wave % 2 * 4 + lane / 16)) * 16u;
  const char* wsrc = reinterpret_cast<const char*>(w) + (static_cast<size_t>(f0) * ktiles + 2 * first) * 1024;
  const char* asrc = reinterpret_cast<const char*>(a) + static_cast<size_t>(t0) * lda * 4 + static_cast<size_t>(first) * 128;
  const unsigned base =
      static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)&mem[0][0])) + wave * 1024;
  auto load = [&](int slot, int stage) {
    const int st = stage < stages ? stage : 0;  // past the end: stage 0 again, never multiplied
#pragma unroll
    for (int u = 0; u < RT; ++u) SHK_LOAD_TO_LDS(base + (slot * (kW + kA) + 4 * u) * 1024, woff[u], wsrc + static_cast<size_t>(st) * 2048);
#pragma unroll
    for (int u = 0; u < CT; ++u) SHK_LOAD_TO_LDS(base + (slot * (kW + kA) + kW + 4 * u) * 1024, aoff[u], asrc + static_cast<size_t>(st) * 128);
  };

  mf4 acc[RT][CT], group[RT][CT], total[RT][CT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[r][c] = group[r][c] = total[r][c] = mf4{0.f, 0.f, 0.f, 0.f};
  int in_seg = 0, in_group = 0;
  load(0, 0);
  load(1, 1);
  int slot = 0;
  for (int st = 0; st < stages; ++st) {
    SHK_MEET_WITH_LOADS(RT + CT);
    load(slot ? slot - 1 : kRing - 1, st + 2);
    const mf4(*now)[kWave] = mem + slot * (kW + kA);
    mf4 wv[2][RT], av[2][CT];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int r = 0; r < RT; ++r) wv[half][r] = now[(mw * RT + r) * 2 + half][lane];
#pragma unroll
      for (int c = 0; c < CT; ++c)  // row i of 16: unit i / 8, its row i % 8
        av[half][c] = now[kW + (nw * CT + c) * 2 + i / 8][i % 8 * 8 + ((half * 4 + kg) ^ (i / 2))];
    }
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int c = 0; c < CT; ++c)
            acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[half][r][j], av[half][c][j], acc[r][c], 0, 0, 0);
      if (++in_seg == seg_steps) {  // a segment ends
        in_seg = 0;
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int c = 0; c < CT; ++c) {
            group[r][c] += acc[r][c];
            acc[r][c] = mf4{0.f, 0.f, 0.f, 0.f};
          }
        if (++in_group == kF32Group) {
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
    }
    slot = slot + 1 < kRing ? slot + 1 : 0;
  }
  SHK_WAIT_LOADS(0);  // no load may arrive in LDS that the workgroup has given back

  if constexpr (GATED) {
    __syncthreads();
#pragma unroll
    for (int c = 0; c < CT; ++c) mem[(mw * 2 + nw) * CT + c][lane] = total[0][c] + (group[0][c] + acc[0][c]);
    __syncthreads();
    const int row = threadIdx.x / 4, quad = threadIdx.x % 4;  // four neighbouring threads a row's 64 bytes
    if (row >= 32 * CT || t0 + row >= n) return;
    const mf4 g = mem[row / 16][quad * 16 + row % 16], up = mem[2 * CT + row / 16][quad * 16 + row % 16];
    mf4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = f32_gate(g[e], up[e], gate);
    float* dst = out + static_cast<size_t>(t0 + row) * ldo + f0 * 16 + quad * 4;
    if (vec_out) {
      *reinterpret_cast<mf4*>(dst) = v;
    } else {  // (out does not begin at a multiple of 16 bytes)
#pragma unroll
      for (int e = 0; e < 4; ++e) dst[e] = v[e];
    }
    return;
  }
  if (GROUPS) out += static_cast<size_t>(blockIdx.y) * n * ldo;
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    const int row = t0 + (nw * CT + c) * 16 + i;  // the matrix instruction's columns
    if (row >= n) continue;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const int col = (f0 + mw * RT + r) * 16 + kg * 4;
      mf4 v = total[r][c] + (group[r][c] + acc[r][c]);
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
}

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

template <int RT, int CT, bool GATED = false, bool GROUPS = false>
static void launch_f32_lds(const F32Product& p, hipStream_t s, F32Gate gate = F32Gate{}) {
  constexpr int F = GATED ? 16 : 32 * RT;
  const int tiles = (p.m + F - 1) / F * ((p.n + 32 * CT - 1) / (32 * CT));
  const int vec_out = p.ldo % 4 == 0 && reinterpret_cast<uintptr_t>(p.out) % 16 == 0;
  const dim3 grid((tiles + kDies - 1) / kDies * kDies, GROUPS ? kF32Segments / kF32Group : 1);
  gemm_f32_lds_kernel<RT, CT, GATED, GROUPS><<<grid, 4 * kWave, 0, s>>>(p.a, p.w, p.bias, p.out, p.n, p.m, p.k, p.lda, p.ldo, p.accumulate,
                                                                        vec_out, gate);
}

// Sizes for which gemm_f32_few_kernel is the faster one.  Weights cold, gemm_f32_kernel and it, us at 1 / 8 / 16 rows: half blocks and
// segments as long as a wavefront holds its steps (2048 x 2048 7.7 / 8.6 / 10.3 and 7.0 / 7.1 / 8.8, x 4096 11.7 / 12.3 / 14.7 and 14.9 / 16.6 /
// 19.6); up to 8,192 features (8192 x 4096 32.5 / 33.4 / 42.0 and 26.5 / 27.3 / 32.2); with more of them whole blocks of a long k are a part of
// a second round (11008 x 2048 19.0 / 19.7 / 23.7 and 21.4 / 23.5 / 28.0, 32000 x 2048 40.7 / 40.2 / 43.9 and 52.3 / 60.0 / 71.4; x 1024 11.8 /
// 12.3 / 14.5 and 9.6 / 10.4 / 12.3), and with still more the kernel above has rounds enough (16384 x 512 8.9 / 9.1 / 10.3 and 8.9 / 9.2 / 10.3,
// x 896 12.8 / 13.0 / 14.4 and 12.2 / 12.4 / 15.8, 50000 x 256 12.6 / 12.7 / 13.7 and 18.7 / 20.8 / -, x 1024 35.6 / 35.8 / 36.1 and 32.1 /
// 34.2 / -; 151936 x 896 98 / - / 107 and 90 / - / 121).
static bool f32_few(int n, int m, int k) {
  if (n > 16 || k % 16) return false;
  if (m <= 2048) return k <= 2560;
  if (m <= 8192) return true;
  if (m <= 12288) return k <= 1024;
  return n <= 8 && k >= 896 && k <= 1024;
}

// Half blocks of features and a segment a wavefront up to 2,048 features, the segments also for a k of up to 1,024, else a group
// a wavefront: 9728 x 896 at 4 rows 8.7 us by segments, 10.0 by groups, 3584 x 3584 15.5 and 12.2, 3584 x 18944 at 16 rows 70 and 61.
static void launch_f32_few(const F32Product& p, hipStream_t s) {
  const int seg_steps = (p.k + 16 * kF32Segments - 1) / (16 * kF32Segments);
  if (p.m <= 2048) {  // (a k of up to 2,560: ten steps)
    if (seg_steps <= 2) run_f32_few<16, 8, 2, false, false>(p, s);
    else if (seg_steps <= 4) run_f32_few<16, 8, 4, false, false>(p, s);
    else if (seg_steps <= 6) run_f32_few<16, 8, 6, false, false>(p, s);
    else run_f32_few<16, 8, 10, false, false>(p, s);
  } else if (p.k <= 1024) {  // (four steps)
    if (seg_steps <= 2) run_f32_few<16, 16, 2, false, false>(p, s);
    else run_f32_few<16, 16, 4, false, false>(p, s);
  } else {
    run_f32_few<4, 16, 0, false, false>(p, s);
  }
}

// The shape of the kernel for a size (results are the same bits in all of them).  Measured on the 0.5B
// model's matrices, tiled weights, microseconds:
//   up to 16 rows (what f32_few() leaves; 896 x 896 and 9728 x 896 are here for rows that are not aligned, or a k that is no multiple of
//     16): 896 x 896 5 in one-tile workgroups of 16 segments (9 with four row blocks and four groups of
//     k), 896 x 4864 13 (37); 9728 x 896 10.7 with four row blocks (12), 151936 x 896 98 with eight (113);
//   more: the largest tile that still leaves the 256 compute units evenly loaded.  896 x 896 at 64 / 128 / 509 /
//     1024 rows 5.7 / 7.3 / 17 / 26 (16 x 16, 32 x 16, 32 x 64, 64 x 64), 9728 x 896 at 64 / 509 25 / 124
//     (32 x 32, 64 x 64: 70 TFLOP/s of the 150 that the instruction reaches alone).  A k of up to 256 is one step
//     a segment, and a shorter one leaves the later of four groups without any: there a wavefront walks all of k and
//     four lie side by side along the rows.
//     1,501 rows: 28 products of 448 x 128 160 us shared by four groups, 77 so
//     (95 with vector instructions), 14 of 128 x 64 27, 13 (14), 40 of 256 x 192 132, 86 (105), 4864 x 256 73, 55 (66).
//   tiled weights of a k in whole stages, enough of them: gemm_f32_lds_kernel with 32 features x 64 rows, or 32 x 32 where those
//     are few and k is short.  9728 x 896 at 64 / 200 / 509 / 1,024 rows 18.8 / 45.7 / 91.8 / 163 (24 / 62.6 / 120.6 / 229.5
//     without it), 1152 x 896 at 509 / 2,000 18.7 / 43.9 (23.7 / 63.1), 3584 x 3584 at 1,501 325 (414), 896 x 4864 at 1,024 97.7
//     (100.8), but at 509 (224 workgroups of 32 x 64) 61 against 57, 1152 x 896 at 200 (252 of 32 x 32) 10.7 against 9.3.
template <bool TILED>
static void run_f32(const F32Product& p, hipStream_t s) {
  auto tiles = [&](int rows, int cols) {
    return static_cast<long long>((p.m + rows - 1) / rows) * ((p.n + cols - 1) / cols) * p.batch;
  };
  auto one_round = [](long long count) { return count >= 192 && count <= 256; };
  // whole stages of aligned rows, offsets within a tile of 32 bits
  const bool staged = TILED && p.batch == 1 && p.k % 32 == 0 && p.k > 256 && p.k <= 1 << 20 && p.lda % 4 == 0 && p.lda <= 1 << 20 &&
                      reinterpret_cast<uintptr_t>(p.a) % 16 == 0;
  const bool few = TILED && f32_few(p.n, p.m, p.k) && p.lda % 4 == 0 && reinterpret_cast<uintptr_t>(p.a) % 16 == 0;
  if (few) {
    launch_f32_few(p, s);
  } else if (p.n <= 16) {
    if (p.m <= 2048)
      launch_f32<1, 1, 16, 1, 1, 2, TILED>(p, s);
    else if (p.m <= 32768)
      launch_f32<1, 1, 4, 4, 1, 4, TILED>(p, s);
    else
      launch_f32<2, 1, 4, 4, 1, 2, TILED>(p, s);
  } else if (staged && (tiles(32, 64) >= 1536 || (p.k > 1024 && tiles(32, 64) >= 440))) {
    launch_f32_lds<1, 2>(p, s);
  } else if (staged && p.k <= 1024 && tiles(32, 32) > kDies * 32) {
    launch_f32_lds<1, 1>(p, s);
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

// Sizes for which gemm_f32_lds_kernel forms groups (from a k of 768 on: none of them is empty) and gated products: whole stages, a
// matrix's offsets of 32 bits.
static bool f32_staged(int m, int k, int lda) {
  return k % 32 == 0 && k > 256 && lda <= 1 << 20 && static_cast<long long>(m) * k < 1LL << 30;
}

// Groups in which shk_gemm_f32_groups may leave a product for its reader (1: only whole): four where a long k would be walked in few
// workgroups.
extern "C" int shk_gemm_f32_splits(int n, int m, int k) {
  const long long tiles = (m + 31LL) / 32 * ((n + 63) / 64);
  const bool few = n <= 16 && m <= 2048 && k >= 2048 && k % 16 == 0, more = n >= 64 && k >= 4096 && tiles <= 640 && f32_staged(m, k, k);
  return m % 4 == 0 && (few || more) ? kF32Segments / kF32Group : 1;
}

// Whether the groups and a norm that adds them are faster than the product whole and the norm.  Weights cold, us, whole -> in groups.
// Up to 16 rows, at 1 / 8 / 16: 896 x 4864 14.8 / 16.1 / 18.3 -> 11.4 / 12.0 / 13.9, 1024 x 16384 34.7 / 36.3 / 42.6 -> 24.0 / 24.7 / 31.6; with more features the
// product has workgroups enough but for steps that its wavefronts hold at once: 1536 x 2560 9.5 / 9.9 / 12.0 -> 9.1 / 9.4 / 11.0, x 2576 11.3 / 12.0 /
// 12.5 -> 13.0 / 13.8 / 16.9, x 8960 23.3 / 24.6 / 28.0 -> 22.2 / 24.3 / 29.1, 2048 x 2048 9.9 / 10.2 / 11.9 -> 10.2 / 10.6 / 12.4, x 5632 17.2 / 18.2 /
// 21.0 -> 21.7 / 22.3 / 29.1 (1024 x 2576 10.9 / 11.6 / 12.0 -> 10.4 / 10.9 / 13.0).
// More rows, at 64 / 100 / 256 / 512 / 1,000 / 2,000: 896 x 4864 19.3 / 27.2 / 33.5 / 58.4 / 97 / 179 -> 20.2 / 20.9 / 30.7 / 49.5 / 83 / 171, 1536 x 8960
// 42.9 / 53.7 / 94.7 / 173 / 251 / 484 -> 32.3 / 48.5 / 67.8 / 123 / 233 / 479 (up to 640 workgroups a group); tiles of 16 x 16 that the chip holds at once share
// k among sixteen wavefronts: 256 x 4096 at 64 / 256 / 512 15.7 / 16.0 / 22.9 -> 17.2 / 17.7 / 18.6.  A short k gains nothing: 512 x 2048 at 64 / 320
// 11.2 / 16.8 -> 11.9 / 16.8.
extern "C" int shk_gemm_f32_groups_faster(int n, int m, int k) {
  if (shk_gemm_f32_splits(n, m, k) == 1) return 0;
  if (n <= 16) return m <= 1536 && (k <= 2560 || (k >= 4096 && (m <= 1024 || n <= 8)));
  return (m + 15LL) / 16 * ((n + 15) / 16) > 256;
}

extern "C" int shk_gemm_f32_groups(const void* a, const void* wt, void* out, int n, int m, int k, int lda, void* stream) {
  SHK_REQUIRE(n >= 0 && m > 0 && k > 0 && k % 16 == 0 && lda >= k && lda % 4 == 0 && (n <= 16 || (k >= 768 && f32_staged(m, k, lda))),
              "gemm_f32_groups: bad sizes n=%d m=%d k=%d lda=%d", n, m, k, lda);
  if (n == 0) return 0;
  SHK_REQUIRE(a && wt && out && reinterpret_cast<uintptr_t>(wt) % 16 == 0 && reinterpret_cast<uintptr_t>(a) % 16 == 0,
              "gemm_f32_groups: null or misaligned pointer");
  const F32Product p{static_cast<const float*>(a), static_cast<const float*>(wt), nullptr, static_cast<float*>(out), n, m, k, lda, m, 0, 1, 0, 0, 0};
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (n <= 16) {  // (ten steps a segment are asked for at once, which is a k of 2,560)
    if (k <= 2560) run_f32_few<4, 8, 10, false, true>(p, s);
    else run_f32_few<4, 8, 0, false, true>(p, s);
  } else {
    launch_f32_lds<1, 2, false, true>(p, s);
  }
  SHK_LAUNCH_CHECK("gemm_f32_groups");
  return 0;
}

// Whether shk_gemm_f32_gated takes a product of 2 m features, gate and other factor.
extern "C" int shk_gemm_f32_gated_takes(int n, int m, int k) {
  return m > 0 && m % 16 == 0 && k > 0 && k % 16 == 0 && (n <= 16 || f32_staged(m, k, k));
}

// Whether it is faster than product and gate in two kernels.  Weights cold, us, two kernels -> one.
// Up to 16 rows, at 1 / 16: a k of up to 1,024 (segments a wavefront) always, 4864 x 896 13.0 / 15.7 -> 11.3 / 13.5, 256 x 896 6.3 / 7.8 -> 5.4 /
// 7.1.  A longer one is walked in four groups, by one workgroup a compute unit: up to 1,024 features the product alone has half blocks and
// sixteen segments (768 x 2048 9.0 / 10.5 -> 12.1 / 14.2), up to 4,096 it has not (1040 x 2048 19.9 / 24.7 -> 12.7 / 14.5, 4096 x 2048 21.0 /
// 25.8 -> 15.9 / 18.6); from there on whole blocks are a part of a second round (4480 x 2048 21.0 / 25.6 -> 24.0 / 28.6, 8192 x 2048 24.8 / 26.6 ->
// 28.3 / 31.8) until it is the product that begins its second (8448 x 2048 38.3 / 45.1 -> 33.9 / 41.8, 11008 x 4096 80.5 / 95.9 -> 66.7 / 77.2;
// 12288 x 2048 39.0 / 45.5 -> 40.8 / 46.2, 13056 x 2048 39.4 / 46.0 -> 48.4 / 55.8).
// More rows, whose k one workgroup walks whole where the product shares it among wavefronts: as many workgroups of 32 rows as compute
// units, unless k is shorter.  4864 x 896 at 17 / 64 / 128 / 509 / 2,000 16.5 / 20.6 / 29.5 / 88.1 / 356 -> 14.2 / 17.8 / 26.9 / 83.2 / 346, 8960 x 1536
// at 17 / 509 49.6 / 250 -> 30.7 / 247, 512 x 288 6.2 / 9.3 -> 5.4 / 7.0; 768 x 2048 at 17 / 128 10.8 / 16.7 -> 18.6 / 19.2, at 256 28.1 -> 26.4;
// 2816 x 2048 at 17 / 33 17.3 / 31.0 -> 19.5 / 26.8; 256 x 512 at 17 8.1 -> 7.7, 768 x 896 at 128 11.3 -> 10.5, at 65 9.7 -> 10.6.
static bool f32_gated_faster(int n, int m, int k) {
  if (!shk_gemm_f32_gated_takes(n, m, k)) return false;
  if (n <= 16) return k <= 1024 || (m > 1024 && m <= 4096) || (m > 8192 && m <= 11264);
  const long long groups = m / 16 * ((n + 31LL) / 32);
  return k <= 512 || groups > 256 || (k <= 896 && groups >= 176);
}

extern "C" int shk_gemm_f32_gated_faster(int n, int m, int k) { return f32_gated_faster(n, m, k); }

extern "C" int shk_gemm_f32_gated(const void* a, const void* wt, void* out, int n, int m, int k, int lda, int act, float limit,
                                  float up_shift, void* stream) {
  SHK_REQUIRE(n >= 0 && m > 0 && m % 16 == 0 && k > 0 && k % 16 == 0 && lda >= k && lda % 4 == 0 && (n <= 16 || f32_staged(m, k, lda)),
              "gemm_f32_gated: bad sizes n=%d m=%d k=%d lda=%d", n, m, k, lda);
  SHK_REQUIRE(act >= 1 && act <= 4 && limit >= 0.f, "gemm_f32_gated: unknown gate");
  if (n == 0) return 0;
  SHK_REQUIRE(a && wt && out && reinterpret_cast<uintptr_t>(wt) % 16 == 0 && reinterpret_cast<uintptr_t>(a) % 16 == 0,
              "gemm_f32_gated: null or misaligned pointer");
  const int seg_steps = (k + 16 * kF32Segments - 1) / (16 * kF32Segments);
  const F32Gate gate = {act, limit, up_shift};
  if (n > 16) {
    const F32Product p{static_cast<const float*>(a), static_cast<const float*>(wt), nullptr, static_cast<float*>(out), n, m, k, lda, m, 0, 1, 0, 0, 0};
    const long long tiles = m / 16 * ((n + 63LL) / 64);
    // (as for the product whole, but for a long k only where the last round of two workgroups a compute unit is at least half full: 32 and 64
    // rows a workgroup, 1536 x 4096 at 512 rows (768 tiles of 64) 122 and 116 us, 14336 x 2048 at 64 (896) 78 and 70, 4864 x 2048 at 128 (608)
    // 52 and 57, 8960 x 2048 at 64 (560) 51 and 57)
    if (tiles >= 1536 || (k > 1024 && n > 32 && tiles >= 440 && (tiles + 256) % 512 <= 256))
      launch_f32_lds<1, 2, true>(p, static_cast<hipStream_t>(stream), gate);
    else
      launch_f32_lds<1, 1, true>(p, static_cast<hipStream_t>(stream), gate);
    SHK_LAUNCH_CHECK("gemm_f32_gated");
    return 0;
  }
  const F32Product p{static_cast<const float*>(a), static_cast<const float*>(wt), nullptr, static_cast<float*>(out), n, m, k, lda, m, 0, 1, 0, 0, 0};
  const hipStream_t few = static_cast<hipStream_t>(stream);
  if (k > 1024) run_f32_few<4, 16, 0, true, false>(p, few, gate);
  else if (seg_steps <= 2) run_f32_few<16, 16, 2, true, false>(p, few, gate);
  else run_f32_few<16, 16, 4, true, false>(p, few, gate);  // (up to four steps a segment)
  SHK_LAUNCH_CHECK("gemm_f32_gated");
  return 0;
}

extern "C" int shk_gemm_f32_few(int n, int m, int k) { return f32_few(n, m, k); }

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
