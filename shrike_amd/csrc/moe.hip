// A routed mixture of gated feed-forward experts.
//
//   scores s = softmax(router logits) over all experts (float32);
//   the `top` experts with the largest s + correction are chosen (the lowest index wins a tie),
//   where the experts form groups only from those of the `keep` groups (of neighbours, of equal
//   size) whose largest s + correction is largest;
//   their weights are their s divided by the chosen experts' sum (+ 1e-20), times `scale`;
//   out = sum over the chosen of weight * W_down_e (act(W_gate_e x) * (W_up_e x + shift))  (+ what a
//   shared expert gave, times sigmoid of a number per token where the design gates it); with a
//   limit the gate's product is bounded from above and the other one from both sides first.
//   Router outputs from `experts` on are identity experts: they have no matrices, their output is x.
//   Experts without a gate whose activation is the square of ReLU are the same with ReLU as act and
//   their one matrix in both places: relu(u) * u; the kernels then form that product once.
//
// moe_route_kernel     a wavefront per token
// moe_gate_up_kernel   a workgroup per (token, chosen expert, block of features): every
//                      (token, expert) pair is a product of its own, summed in one fixed
//                      order, so a token's result does not depend on what else is in the step
// moe_down_kernel      a workgroup per (token, block of columns): the chosen experts'
//                      outputs, weighted and added in the order they were chosen
//
// On the matrix units (bfloat16, many tokens): the (token, expert) pairs are listed per expert
// in the order of the tokens (moe_lists_kernel, a workgroup per expert), and the two products
// run per expert over its list (v_mfma_f32_16x16x32_bf16): short lists in tiles of 32 pairs, operands
// straight from memory, longer ones in tiles of 128 pairs through LDS.  Matrices whose sides are multiples
// of 64 lie in tiles of 16 rows x 32, others row-major with k innermost.  Workgroups beyond
// an expert's list leave at once or take none, so the grid depends on the step's size alone.  A pair's
// sums run over k in one fixed order wherever the pair stands in its list; the pairs' outputs
// are kept in float32 and joined per token in the order the experts were chosen.
#include "api.h"
#include "common.h"
#include "gemm_wide.h"

#include <type_traits>

namespace shk {

// kMaxExpertsPerLane: 1 for up to 64 outputs, 8 for up to 512.
template <int kMaxExpertsPerLane>
__global__ void __launch_bounds__(256)
    moe_route_kernel(const float* __restrict__ logits, int ld, const float* __restrict__ correction, int experts,
                     int top, int groups, int keep, float scale, int32_t* __restrict__ chosen,
                     float* __restrict__ weights, int n) {
  const int t = blockIdx.x * (256 / kWave) + threadIdx.x / kWave;
  const int lane = threadIdx.x % kWave;
  if (t >= n) return;
  float s[kMaxExpertsPerLane], c[kMaxExpertsPerLane];
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < kMaxExpertsPerLane; ++i) {
    const int e = lane + i * kWave;
    s[i] = e < experts ? logits[static_cast<size_t>(t) * ld + e] : -INFINITY;
    mx = fmaxf(mx, s[i]);
  }
  mx = wave_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < kMaxExpertsPerLane; ++i) {
    const int e = lane + i * kWave;
    s[i] = e < experts ? expf(s[i] - mx) : 0.f;
    sum += s[i];
  }
  sum = wave_sum(sum);
#pragma unroll
  for (int i = 0; i < kMaxExpertsPerLane; ++i) {
    const int e = lane + i * kWave;
    s[i] /= sum;
    c[i] = e < experts ? s[i] + (correction ? correction[e] : 0.f) : -INFINITY;
  }
  if (keep < groups) {
    // lane g keeps the best choice score of group g; the `keep` best groups stay, of equal ones the lowest
    const int size = experts / groups;
    float group_best = -INFINITY;
    for (int g = 0; g < groups; ++g) {
      float b = -INFINITY;
#pragma unroll
      for (int i = 0; i < kMaxExpertsPerLane; ++i) {
        const int e = lane + i * kWave;
        if (e >= g * size && e < (g + 1) * size) b = fmaxf(b, c[i]);
      }
      b = wave_max(b);
      if (lane == g) group_best = b;
    }
    unsigned long long kept = 0;
    for (int k = 0; k < keep; ++k) {
      const bool open = lane < groups && !((kept >> lane) & 1ull);
      const float best = wave_max(open ? group_best : -INFINITY);
      unsigned long long at = __ballot(open && group_best == best);
      if (at == 0) at = __ballot(open);  // (scores that are not numbers: the lowest group left)
      kept |= at & (~at + 1ull);
    }
#pragma unroll
    for (int i = 0; i < kMaxExpertsPerLane; ++i) {
      const int e = lane + i * kWave;
      if (e < experts && !((kept >> (e / size)) & 1ull)) c[i] = -INFINITY;
    }
  }
  float picked_sum = 0.f, my_score = 0.f;
  int my_expert = 0;
  for (int k = 0; k < top; ++k) {
    // the largest choice score not yet taken; of equal ones the lowest index
    float best = -INFINITY;
    int best_e = 1 << 30;
#pragma unroll
    for (int i = 0; i < kMaxExpertsPerLane; ++i) {
      const int e = lane + i * kWave;
      if (c[i] > best) {  // ascending e within a lane: the first of equal ones stays
        best = c[i];
        best_e = e;
      }
    }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
      const float ob = __shfl_xor(best, off, kWave);
      const int oe = __shfl_xor(best_e, off, kWave);
      if (ob > best || (ob == best && oe < best_e)) {
        best = ob;
        best_e = oe;
      }
    }
    if (best_e >= experts) {
      // no score compares (logits that are not numbers): the lowest expert not yet taken, so
      // that what is written is always an expert's index
      best_e = 1 << 30;
#pragma unroll
      for (int i = 0; i < kMaxExpertsPerLane; ++i) {
        const int e = lane + i * kWave;
        if (e < experts && !(c[i] == -INFINITY) && e < best_e) best_e = e;
      }
#pragma unroll
      for (int off = kWave / 2; off > 0; off >>= 1) {
        const int oe = __shfl_xor(best_e, off, kWave);
        best_e = oe < best_e ? oe : best_e;
      }
      if (best_e >= experts) best_e = k;  // (cannot happen while top <= experts)
    }
    float score = 0.f;
#pragma unroll
    for (int i = 0; i < kMaxExpertsPerLane; ++i) {
      if (lane + i * kWave == best_e) {
        score = s[i];
        c[i] = -INFINITY;
      }
    }
    score = wave_sum(score);  // one lane holds it
    picked_sum += score;
    if (lane == k) {  // lane k keeps the k-th choice
      my_expert = best_e;
      my_score = score;
    }
  }
  if (lane < top) {
    chosen[static_cast<size_t>(t) * top + lane] = my_expert;
    weights[static_cast<size_t>(t) * top + lane] = my_score / (picked_sum + 1e-20f) * scale;
  }
}

// What joins an expert's two products: the gate's activation, the bound (0: none), what is added to the
// other factor.
struct GateForm {
  int act;
  float limit, shift;
};

__device__ __forceinline__ float gate_act(float g, int act) {
  if (act == 3) return fmaxf(g, 0.f);  // ReLU; with the gate's matrix also the other factor's, the square of ReLU
  if (act == 4) return g / (1.f + expf(-1.702f * g));
  const float x = act == 2 ? 2.f * 0.7978845608028654f * (g + 0.044715f * g * g * g) : g;
  return g / (1.f + expf(-x));
}

__device__ __forceinline__ float gate_times_up(float g, float u, GateForm form) {
  if (form.limit > 0.f) {
    g = fminf(g, form.limit);
    u = fminf(fmaxf(u, -form.limit), form.limit);
  }
  return gate_act(g, form.act) * (u + form.shift);
}

// What multiplies the shared expert's output for token t: sigmoid(add_gate[t * gate_ld]), one number
// per token, or 1 without such a gate.
__device__ __forceinline__ float shared_share(const float* __restrict__ add_gate, int gate_ld, int t) {
  return add_gate ? 1.f / (1.f + expf(-add_gate[static_cast<size_t>(t) * gate_ld])) : 1.f;
}

constexpr int kMoeFeatures = 32;  // features (or columns) a workgroup

template <typename T>
__global__ void __launch_bounds__(256)
    moe_gate_up_kernel(const T* __restrict__ x, const int32_t* __restrict__ chosen, const T* __restrict__ wg,
                       const T* __restrict__ wu, T* __restrict__ act_out, int width, int ff, int top, GateForm form,
                       int experts) {
  extern __shared__ float xs[];
  const int pair = blockIdx.y, t = pair / top;
  const int e = max(chosen[pair], 0);
  if (e >= experts) return;  // an identity expert (an index from memory never leaves the stack of experts)
  for (int k = threadIdx.x; k < width; k += 256) xs[k] = to_float(x[static_cast<size_t>(t) * width + k]);
  __syncthreads();
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  for (int i = wave; i < kMoeFeatures; i += 256 / kWave) {
    const int f = blockIdx.x * kMoeFeatures + i;
    if (f >= ff) break;
    const T* gr = wg + (static_cast<size_t>(e) * ff + f) * width;
    const T* ur = wu + (static_cast<size_t>(e) * ff + f) * width;
    float g = 0.f, u = 0.f;
    if (wg == wu) {  // experts without a gate: the one product is both factors
      for (int k = lane; k < width; k += kWave) g = fmaf(to_float(gr[k]), xs[k], g);
      g = u = wave_sum(g);
    } else {
      for (int k = lane; k < width; k += kWave) {
        g = fmaf(to_float(gr[k]), xs[k], g);
        u = fmaf(to_float(ur[k]), xs[k], u);
      }
      g = wave_sum(g);
      u = wave_sum(u);
    }
    if (lane == 0) act_out[static_cast<size_t>(pair) * ff + f] = from_float<T>(gate_times_up(g, u, form));
  }
}

template <typename T>
__global__ void __launch_bounds__(256)
    moe_down_kernel(const T* __restrict__ x, const T* __restrict__ act_in, const int32_t* __restrict__ chosen,
                    const float* __restrict__ weights, const T* __restrict__ wd, const T* __restrict__ add,
                    const float* __restrict__ add_gate, int gate_ld, T* __restrict__ out, int width, int ff, int top,
                    int experts) {
  extern __shared__ float as[];  // [top, ff]
  const int t = blockIdx.y;
  for (int i = threadIdx.x; i < top * ff; i += 256) as[i] = to_float(act_in[static_cast<size_t>(t) * top * ff + i]);
  __syncthreads();
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  for (int i = wave; i < kMoeFeatures; i += 256 / kWave) {
    const int c = blockIdx.x * kMoeFeatures + i;
    if (c >= width) break;
    float total = 0.f;
    for (int k = 0; k < top; ++k) {
      const int e = max(chosen[static_cast<size_t>(t) * top + k], 0);
      if (e >= experts) {  // an identity expert
        total = fmaf(weights[static_cast<size_t>(t) * top + k], to_float(x[static_cast<size_t>(t) * width + c]), total);
        continue;
      }
      const T* dr = wd + (static_cast<size_t>(e) * width + c) * ff;
      float d = 0.f;
      for (int f = lane; f < ff; f += kWave) d = fmaf(to_float(dr[f]), as[k * ff + f], d);
      total = fmaf(weights[static_cast<size_t>(t) * top + k], wave_sum(d), total);
    }
    if (lane == 0) {
      if (add) total += shared_share(add_gate, gate_ld, t) * to_float(add[static_cast<size_t>(t) * width + c]);
      out[static_cast<size_t>(t) * width + c] = from_float<T>(total);
    }
  }
}

typedef __bf16 mbf16x8 __attribute__((ext_vector_type(8)));
typedef float mf32x4 __attribute__((ext_vector_type(4)));

// order[e * n + r] = the r-th pair (token * top + place among the token's choices) of expert e,
// tokens ascending; counts[e] = how many there are
__global__ void __launch_bounds__(256)
    moe_lists_kernel(const int32_t* __restrict__ chosen, int n, int top, int32_t* __restrict__ order,
                     int32_t* __restrict__ counts) {
  __shared__ int wave_total[256 / kWave];
  const int e = blockIdx.x;
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  int base = 0;
  for (int t0 = 0; t0 < n; t0 += 256) {
    const int t = t0 + threadIdx.x;
    int hit = -1;
    if (t < n)
      for (int k = top - 1; k >= 0; --k)
        if (chosen[static_cast<size_t>(t) * top + k] == e) hit = k;
    const unsigned long long votes = __ballot(hit >= 0);
    const int before = __popcll(votes & ((1ull << lane) - 1ull));
    if (lane == 0) wave_total[wave] = __popcll(votes);
    __syncthreads();
    int prefix = 0, total = 0;
    for (int w = 0; w < 256 / kWave; ++w) {
      if (w < wave) prefix += wave_total[w];
      total += wave_total[w];
    }
    if (hit >= 0) order[static_cast<size_t>(e) * n + base + prefix + before] = t * top + hit;
    base += total;
    __syncthreads();
  }
  if (threadIdx.x == 0) counts[e] = base;
}

// The two products for lists of few pairs, where what counts is how fast the experts' matrices stream: a
// workgroup takes 32 pairs and 32 weight rows (of both matrices where there is a gate), its four wavefronts
// a quarter of k each, so that even one token's experts are read by hundreds of wavefronts; a lane asks for
// four steps' operands at once.  The quarters' sums meet in LDS and are added in order.  The weights' stream is
// what bounds it: with row-major weights (16 pieces of 64 bytes a load) eight tokens' experts (two of eight, 4736
// features of width 3584) took 99 and 56 us, in tiles 83 and 45 (680 MB: 113 us at the memory's rate).
constexpr int kQuarters = 4;

// acc[m][a][b] += W_m[row b] . x[pair a] over this wavefront's quarter of k.  TILED: the weights lie in tiles of
// 16 rows x 32 k (512 elements; wr points at the lane's 8 of the row block's first tile), one run of 1 KiB a load
template <int MATRICES, bool TILED>
__device__ __forceinline__ void moe_quarter(const bf16* const (&xr)[2], const bool (&have_pair)[2],
                                            const bf16* const (&wr)[MATRICES][2], int k, int quarter, int kg,
                                            mf32x4 (&acc)[MATRICES][2][2]) {
  constexpr int kAhead = 4;
  const int per = (k + 32 * kQuarters - 1) / (32 * kQuarters) * 32;
  const int begin = quarter * per, end = begin + per < k ? begin + per : k;
  for (int k0 = begin; k0 < end; k0 += 32 * kAhead) {
    uint4 av[kAhead][2], wv[kAhead][MATRICES][2];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int kk = k0 + 32 * u;
      const bool have = kk + kg * 8 < end;  // (k is a multiple of 8: a piece is whole or absent)
#pragma unroll
      for (int m = 0; m < MATRICES; ++m)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          wv[u][m][b] = make_uint4(0, 0, 0, 0);
          if (have) wv[u][m][b] = *reinterpret_cast<const uint4*>(wr[m][b] + (TILED ? kk * 16 : kk));
        }
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        av[u][a] = make_uint4(0, 0, 0, 0);
        if (have && have_pair[a]) av[u][a] = *reinterpret_cast<const uint4*>(xr[a] + kk);
      }
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
#pragma unroll
      for (int m = 0; m < MATRICES; ++m)
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
          for (int b = 0; b < 2; ++b)
            acc[m][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(mbf16x8, wv[u][m][b]),
                                                                   __builtin_bit_cast(mbf16x8, av[u][a]), acc[m][a][b], 0, 0, 0);
  }
}

// The quarters' sums of tile (a, b) = (wave / 2, wave % 2) for this wavefront, added in order.
template <int MATRICES>
__device__ __forceinline__ void moe_join_quarters(const mf32x4 (&acc)[MATRICES][2][2], int wave, int lane,
                                                  float4 (&sums)[kQuarters][4][MATRICES][kWave], mf32x4 (&total)[MATRICES]) {
#pragma unroll
  for (int m = 0; m < MATRICES; ++m)
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
        sums[wave][2 * a + b][m][lane] = make_float4(acc[m][a][b][0], acc[m][a][b][1], acc[m][a][b][2], acc[m][a][b][3]);
  __syncthreads();
#pragma unroll
  for (int m = 0; m < MATRICES; ++m) {
    total[m] = mf32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < kQuarters; ++q) {
      const float4 x = sums[q][wave][m][lane];
      total[m][0] += x.x, total[m][1] += x.y, total[m][2] += x.z, total[m][3] += x.w;
    }
  }
}

// act[pair, f] = act(W_gate_e[f] . x_t) * (W_up_e[f] . x_t) for the pairs of expert e's list.  SINGLE: experts
// without a gate, the one product is both factors.
template <bool SINGLE, bool TILED>
__global__ void __launch_bounds__(256)
    moe_gate_up_mfma_kernel(const bf16* __restrict__ x, const int32_t* __restrict__ order,
                            const int32_t* __restrict__ counts, const bf16* __restrict__ wg,
                            const bf16* __restrict__ wu, bf16* __restrict__ act_out, int n, int width, int ff, int top,
                            GateForm form) {
  constexpr int M = SINGLE ? 1 : 2;
  __shared__ float4 sums[kQuarters][4][M][kWave];
  const int e = blockIdx.z;
  const int count = min(counts[e], n);
  const int row0 = blockIdx.y * 32;
  if (row0 >= count) return;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int i = lane % 16, kg = lane / 16;
  const int f0 = blockIdx.x * 32;
  int pair[2];
  bool have[2];
  const bf16* xr[2];
  const bf16* wr[M][2];
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int r = row0 + a * 16 + i;
    pair[a] = r < count ? order[static_cast<size_t>(e) * n + r] : -1;
    have[a] = pair[a] >= 0;
    const int t = have[a] ? min(pair[a] / top, n - 1) : 0;
    xr[a] = x + static_cast<size_t>(t) * width + kg * 8;
    // (in tiles: ff is a multiple of 64)
    const size_t f = static_cast<size_t>(e) * ff + (TILED ? f0 + a * 16 : min(f0 + a * 16 + i, ff - 1));
    const size_t at = f * width + (TILED ? lane * 8 : kg * 8);
    wr[0][a] = wg + at;
    if (!SINGLE) wr[M - 1][a] = wu + at;
  }
  mf32x4 acc[M][2][2], total[M];
#pragma unroll
  for (int m = 0; m < M; ++m)
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) acc[m][a][b] = mf32x4{0.f, 0.f, 0.f, 0.f};
  moe_quarter<M, TILED>(xr, have, wr, width, wave, kg, acc);
  moe_join_quarters<M>(acc, wave, lane, sums, total);
  // features were the rows of the products: this lane holds features f0 + 16 b + 4 kg + r of pair row a * 16 + i
  const int p = wave / 2 ? pair[1] : pair[0];
  if (p < 0) return;
  const int f = f0 + wave % 2 * 16 + 4 * kg;
  bf16* dst = act_out + static_cast<size_t>(p) * ff + f;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (f + r < ff) dst[r] = from_float<bf16>(gate_times_up(total[0][r], total[M - 1][r], form));
}

// pair_out[pair, c] = W_down_e[c] . act[pair]
template <bool TILED>
__global__ void __launch_bounds__(256)
    moe_down_mfma_kernel(const bf16* __restrict__ act_in, const int32_t* __restrict__ order,
                         const int32_t* __restrict__ counts, const bf16* __restrict__ wd,
                         float* __restrict__ pair_out, int n, int width, int ff, int top) {
  __shared__ float4 sums[kQuarters][4][1][kWave];
  const int e = blockIdx.z;
  const int count = min(counts[e], n);
  const int row0 = blockIdx.y * 32;
  if (row0 >= count) return;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int i = lane % 16, kg = lane / 16;
  const int c0 = blockIdx.x * 32;
  int pair[2];
  bool have[2];
  const bf16* ar[2];
  const bf16* wr[1][2];
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int r = row0 + a * 16 + i;
    pair[a] = r < count ? order[static_cast<size_t>(e) * n + r] : -1;
    have[a] = pair[a] >= 0;
    ar[a] = act_in + static_cast<size_t>(have[a] ? min(pair[a], n * top - 1) : 0) * ff + kg * 8;
    wr[0][a] = wd + (static_cast<size_t>(e) * width + (TILED ? c0 + a * 16 : min(c0 + a * 16 + i, width - 1))) * ff +
               (TILED ? lane * 8 : kg * 8);
  }
  mf32x4 acc[1][2][2], total[1];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[0][a][b] = mf32x4{0.f, 0.f, 0.f, 0.f};
  moe_quarter<1, TILED>(ar, have, wr, ff, wave, kg, acc);
  moe_join_quarters<1>(acc, wave, lane, sums, total);
  const int p = wave / 2 ? pair[1] : pair[0];
  if (p < 0) return;
  const int c = c0 + wave % 2 * 16 + 4 * kg;
  float* dst = pair_out + static_cast<size_t>(p) * width + c;
  if (c + 3 < width) {
    *reinterpret_cast<float4*>(dst) = make_float4(total[0][0], total[0][1], total[0][2], total[0][3]);
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (c + r < width) dst[r] = total[0][r];
  }
}

// The same two products for lists of many pairs, tiled through LDS: a workgroup forms 128 pairs x 128
// weight rows (gate/up: 64 features of each; down: 128 columns) in steps of 32 along k.  The four
// wavefronts (2 x 2) take 64 x 64 each: four A and four B operands from LDS feed sixteen matrix
// instructions.  Rows of 32 elements lie 80 bytes apart in LDS, so the sixteen 16-byte reads of an
// operand meet every bank once.  The next step's pieces are fetched into registers while this one is
// multiplied.  Sums run over k in ascending order (in the kernels above, over its quarters).
constexpr int kTileRows = 128;
constexpr int kTileLd = 40;  // elements between rows in LDS (32 and 16 bytes of padding)

// SINGLE (with GATED): the experts have no gate; the tile is 128 features of the one matrix, as in the
// down product, over the tokens' rows, and a feature's product is both factors of its activation.
template <bool GATED, bool SINGLE = false>
__global__ void __launch_bounds__(256)
    moe_tiled_mfma_kernel(const bf16* __restrict__ a, const int32_t* __restrict__ order,
                          const int32_t* __restrict__ counts, const bf16* __restrict__ w0, const bf16* __restrict__ w1,
                          bf16* __restrict__ act_out, float* __restrict__ pair_out, int n, int k, int m, int top, GateForm form) {
  __shared__ __attribute__((aligned(16))) uint16_t sa[2][kTileRows * kTileLd];
  __shared__ __attribute__((aligned(16))) uint16_t sb[2][kTileRows * kTileLd];
  const int e = blockIdx.z;
  const int count = min(counts[e], n);
  const int row0 = blockIdx.y * kTileRows;
  if (row0 >= count) return;
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int i = lane % 16, kg = lane / 16;
  const int wm = wave / 2, wn = wave % 2;
  const int lr = tid / 4, lp = tid % 4;  // the row (and the one 64 below) and the 16-byte piece that this thread stages
  const int32_t* list = order + static_cast<size_t>(e) * n;
  const bf16* arow[2];
  const bf16* brow[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int r = row0 + lr + 64 * h;
    const int pair = r < count ? list[r] : -1;
    // gate/up: a pair's row is its token's; down: its own row of activations
    arow[h] = pair < 0 ? nullptr : a + static_cast<size_t>(GATED ? min(pair / top, n - 1) : min(pair, n * top - 1)) * k + lp * 8;
    if (GATED && !SINGLE) {
      const int f = blockIdx.x * 64 + lr;
      brow[h] = f < m ? (h == 0 ? w0 : w1) + (static_cast<size_t>(e) * m + f) * k + lp * 8 : nullptr;
    } else {
      const int c = blockIdx.x * 128 + lr + 64 * h;
      brow[h] = c < m ? w0 + (static_cast<size_t>(e) * m + c) * k + lp * 8 : nullptr;
    }
  }
  uint4 ra[2], rb[2];
  auto fetch = [&](int k0) {
    const bool have = k0 + lp * 8 < k;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      ra[h] = rb[h] = make_uint4(0, 0, 0, 0);
      if (have && arow[h]) ra[h] = *reinterpret_cast<const uint4*>(arow[h] + k0);
      if (have && brow[h]) rb[h] = *reinterpret_cast<const uint4*>(brow[h] + k0);
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      *reinterpret_cast<uint4*>(&sa[buf][(lr + 64 * h) * kTileLd + lp * 8]) = ra[h];
      *reinterpret_cast<uint4*>(&sb[buf][(lr + 64 * h) * kTileLd + lp * 8]) = rb[h];
    }
  };
  constexpr int kOperands = 4;  // B operands a step
  mf32x4 acc[4][4];
#pragma unroll
  for (int am = 0; am < 4; ++am)
#pragma unroll
    for (int bn = 0; bn < 4; ++bn) acc[am][bn] = mf32x4{0.f, 0.f, 0.f, 0.f};
  fetch(0);
  stage(0);
  __syncthreads();
  int buf = 0;
  for (int k0 = 0; k0 < k; k0 += 32, buf ^= 1) {
    const bool more = k0 + 32 < k;
    if (more) fetch(k0 + 32);
    mbf16x8 af[4], bf[4];
#pragma unroll
    for (int am = 0; am < 4; ++am)
      af[am] = __builtin_bit_cast(mbf16x8, *reinterpret_cast<const uint4*>(&sa[buf][(wm * 64 + am * 16 + i) * kTileLd + kg * 8]));
#pragma unroll
    for (int bn = 0; bn < kOperands; ++bn) {
      // gate/up: operands 0, 1 are this wavefront's 32 gate features, 2, 3 the same features of up (rows 64 on)
      const int brw = GATED && !SINGLE ? (bn / 2) * 64 + wn * 32 + (bn % 2) * 16 + i : wn * 64 + bn * 16 + i;
      bf[bn] = __builtin_bit_cast(mbf16x8, *reinterpret_cast<const uint4*>(&sb[buf][brw * kTileLd + kg * 8]));
    }
#pragma unroll
    for (int am = 0; am < 4; ++am)
#pragma unroll
      for (int bn = 0; bn < kOperands; ++bn)
        acc[am][bn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[bn], af[am], acc[am][bn], 0, 0, 0);
    if (more) stage(buf ^ 1);
    __syncthreads();
  }
  // this lane holds weight rows 4 kg + r of operand bn for the pair in row wm * 64 + am * 16 + i of the tile
#pragma unroll
  for (int am = 0; am < 4; ++am) {
    const int r = row0 + wm * 64 + am * 16 + i;
    if (r >= count) continue;
    const int pair = min(max(list[r], 0), n * top - 1);
    if (GATED && SINGLE) {
      bf16* dst = act_out + static_cast<size_t>(pair) * m;
#pragma unroll
      for (int bn = 0; bn < 4; ++bn) {
        const int f = blockIdx.x * 128 + wn * 64 + bn * 16 + 4 * kg;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (f + q < m) dst[f + q] = from_float<bf16>(gate_times_up(acc[am][bn][q], acc[am][bn][q], form));
      }
    } else if (GATED) {
      bf16* dst = act_out + static_cast<size_t>(pair) * m;
#pragma unroll
      for (int bn = 0; bn < 2; ++bn) {
        const int f = blockIdx.x * 64 + wn * 32 + bn * 16 + 4 * kg;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (f + q < m) dst[f + q] = from_float<bf16>(gate_times_up(acc[am][bn][q], acc[am][bn + 2][q], form));
      }
    } else {
      float* dst = pair_out + static_cast<size_t>(pair) * m;
#pragma unroll
      for (int bn = 0; bn < 4; ++bn) {
        const int c = blockIdx.x * 128 + wn * 64 + bn * 16 + 4 * kg;
        if (c + 3 < m) {
          *reinterpret_cast<float4*>(dst + c) = make_float4(acc[am][bn][0], acc[am][bn][1], acc[am][bn][2], acc[am][bn][3]);
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (c + q < m) dst[c + q] = acc[am][bn][q];
        }
      }
    }
  }
}

// The same two products for weights in tiles (k and m multiples of 64): wide_loop() of gemm_wide.h over a tile of weight rows (gate/up:
// half of them of each) x pairs, 256 x 128, 256 x 192 or 128 x 192.  A unit of the loop's activations is 8 pairs' rows
// x 128 bytes, gathered on the way into LDS, since a lane gives its own address.
// The grid is one row of workgroups and the lists' lengths are only known on the device: workgroup p takes the
// p / 8-th tile of die p % 8's share of all live tiles, counted expert by expert, features outside, the
// expert's pairs inside, so that the 32 compute units of a die read a matrix from memory once and its pairs'
// rows stay in the die's L2.
// What bounds it: as the loop, the multiplications' power limit, the pairs that a list's last tile lacks, and the last round.  1,501 tokens, two of
// eight experts of 4736 features and width 3584: gate/up 213 us, down 99 (262 and 157 with 16 x 16 multiplications and
// a pair's row per lane; 360 and 227 in the kernel above; with row-major weights that loop took 350 and 213).  Pairs'
// rows laid out in tiles first (19 us a layer) changed nothing, nor did leaving out the multiplications
// for the empty half of a list's last tile.

// Tile `index` of all experts' live tiles (features x ceil(count / PAIRS) each): expert, first feature
// tile, first pair; false beyond the last.  `index` < 0 asks for none and returns their number in `total`.
template <int PAIRS>
__device__ __forceinline__ bool moe_tile(const int32_t* counts, int experts, int n, int features, int index, int lane,
                                         int& total, int& e, int& within, int& row_tiles) {
  total = 0;
  for (int e0 = 0; e0 < experts; e0 += kWave) {
    const int mine = e0 + lane < experts ? (min(counts[e0 + lane], n) + PAIRS - 1) / PAIRS : 0;
    int before = mine;  // inclusive prefix over the lanes
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const int up = __shfl_up(before, d, kWave);
      if (lane >= d) before += up;
    }
    const int all = __shfl(before, kWave - 1, kWave);
    if (index >= 0 && index < total + all * features) {
      const int first = total + (before - mine) * features;
      const unsigned long long hit = __ballot(mine > 0 && index >= first && index < first + mine * features);
      const int at = __ffsll(hit) - 1;
      e = e0 + at;
      row_tiles = __shfl(mine, at, kWave);
      within = index - __shfl(first, at, kWave);
      return true;
    }
    total += all * features;
  }
  return false;
}

constexpr int kDieRound = 32;  // workgroups at a time on a die: one a compute unit
enum MoeProduct : int { kMoeGated = 0, kMoeSingle = 1, kMoeDown = 2 };

// One tile of 32 * GM * RM weight rows x 32 * GN * RN pairs of expert e: features f0 and on, the pairs of its list from row0 on.
template <int PRODUCT, int GM, int GN, int RM, int RN>
__device__ __forceinline__ void moe_big_tile(u32x4* mem, int* pairs, int e, int f0, int row0, int count, const bf16* __restrict__ a,
                                             const int32_t* __restrict__ list, const bf16* __restrict__ w0,
                                             const bf16* __restrict__ w1, bf16* __restrict__ act_out,
                                             float* __restrict__ pair_out, int n, int k, int m, int top, GateForm form) {
  using S = WideShape<GM, GN, RM, RN>;
  constexpr int kRows = 32 * GM * RM, kPairs = 32 * GN * RN, kFeatures = PRODUCT == kMoeGated ? kRows / 2 : kRows;
  static_assert(PRODUCT != kMoeGated || S::kWaves % 2 == 0, "a wavefront loads tiles of one of the two matrices");
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  if (threadIdx.x < kPairs) {  // (read behind the loop's barriers)
    const int at = row0 + threadIdx.x;
    pairs[threadIdx.x] = at < count ? min(max(list[at], 0), n * top - 1) : -1;
  }

  // What this wavefront loads: weight tiles and units of 8 pairs wave, wave + kWaves, ..; rows beyond either matrix are read as its
  // last (their products are not stored).  Gated: even tiles are the gate's features, odd ones the same features of up.
  const bool up = PRODUCT == kMoeGated && wave % 2;
  unsigned woff[S::kWLoads], xoff[2 * S::kXLoads];
#pragma unroll
  for (int i = 0; i < S::kWLoads; ++i) {
    const int tile = wave + S::kWaves * i, f = f0 + (PRODUCT == kMoeGated ? tile / 2 : tile) * 16;
    woff[i] = (static_cast<unsigned>((min(f, m - 16) - f0) / 16) * (k / 32) * kWave + lane) * 16u;  // (from row f0 on)
  }
#pragma unroll
  for (int i = 0; i < 2 * S::kXLoads; ++i) {
    const int at = row0 + (wave + S::kWaves * i) * 8 + lane / 8;
    const int pair = max(list[at < count ? at : row0], 0);
    const int row = PRODUCT == kMoeDown ? min(pair, n * top - 1) : min(pair / top, n - 1);
    xoff[i] = static_cast<unsigned>(row) * k * 2u + ((lane % 8) ^ (lane / 8)) * 16u;
  }
  f32x16 acc[RM][RN];
  wide_loop<GM, GN, RM, RN>(acc, mem, reinterpret_cast<const char*>((up ? w1 : w0) + (static_cast<size_t>(e) * m + f0) * k), woff,
                        reinterpret_cast<const char*>(a), xoff, 0u, -1, k / 32, k / 64);

  // Register g * 4 + r of lane (j, half) of a tile of 32 x 32 holds weight row g * 8 + half * 4 + r for pair j.  32 pairs'
  // sums at a time go through LDS and leave in 16-byte pieces along the pairs' rows, several pieces of a lane at a time: a
  // wavefront is alone on its SIMD, so one by one every piece waits for all that it asks for.
  constexpr int kMine = kFeatures / GM;  // output features of a wavefront
  constexpr int kPitch = 32 * RM * 4 + 16, kValues = PRODUCT == kMoeDown ? 4 : 8, kPieces = kMine / kValues;
  const int half = lane / 32, j = lane % 32, first = f0 + wave / GN * kMine;
  char* mine = reinterpret_cast<char*>(mem) + wave * 32 * kPitch;
  auto leave = [&](int jn, auto act) {
#pragma unroll 4
    for (int i = 0; i < 32 * kPieces / kWave; ++i) {
      const int q = i * kWave + lane, t = q / kPieces, row = q % kPieces * kValues, f = first + row;
      const int pair = pairs[(wave % GN * RN + jn) * 32 + t];
      const bool stored = pair >= 0 && f < m;  // (m is a multiple of 64: a piece is inside or outside as a whole)
      const size_t to = static_cast<size_t>(pair) * m + f;
      const float* sums = reinterpret_cast<const float*>(mine + t * kPitch);
      if constexpr (PRODUCT == kMoeDown) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(sums + row);
        if (stored) *reinterpret_cast<f32x4*>(pair_out + to) = v;
      } else {
        const f32x4* gate = reinterpret_cast<const f32x4*>(sums + (PRODUCT == kMoeGated ? row / 16 * 32 + row % 16 : row));
        constexpr int kApart = PRODUCT == kMoeGated ? 4 : 0;
        const GateForm same = {decltype(act)::value, form.limit, form.shift};
        bf16x8 v;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f32x4 g = gate[h], u = gate[kApart + h];
#pragma unroll
          for (int r = 0; r < 4; ++r) v[4 * h + r] = static_cast<__bf16>(gate_times_up(g[r], u[r], same));
        }
        if (stored) *reinterpret_cast<bf16x8*>(act_out + to) = v;
      }
    }
  };
#pragma unroll
  for (int jn = 0; jn < RN; ++jn) {
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4*>(mine + j * kPitch + (i * 32 + g * 8 + half * 4) * 4) =
            f32x4{acc[i][jn][g * 4], acc[i][jn][g * 4 + 1], acc[i][jn][g * 4 + 2], acc[i][jn][g * 4 + 3]};
    SHK_LDS_DONE();
    if (PRODUCT == kMoeDown)
      leave(jn, std::integral_constant<int, 0>{});
    else if (form.act == 4)
      leave(jn, std::integral_constant<int, 4>{});
    else if (form.act == 3)
      leave(jn, std::integral_constant<int, 3>{});
    else if (form.act == 2)
      leave(jn, std::integral_constant<int, 2>{});
    else
      leave(jn, std::integral_constant<int, 1>{});
    SHK_LDS_DONE();
  }
}

// Tiles beyond a die's last whole round of 32 that fill no more than half of one run as two halves of their weight rows each, which take
// little more than half as long: 1,036 tiles of gate and up (1,501 tokens, two of eight experts of 4736 features and width 3584) 231 us ->
// 213, of five rounds; 999 tiles, four rounds with 29 of 32 compute units in the last, 187 either way.
template <int PRODUCT, int GM, int GN, int RM, int RN>
__global__ void __launch_bounds__(GM* GN* kWave) __attribute__((amdgpu_waves_per_eu(GM * GN / 4, GM * GN / 4)))
    moe_big_mfma_kernel(const bf16* __restrict__ a, const int32_t* __restrict__ order,
                        const int32_t* __restrict__ counts, const bf16* __restrict__ w0, const bf16* __restrict__ w1,
                        bf16* __restrict__ act_out, float* __restrict__ pair_out, int n, int k, int m, int experts, int top,
                        GateForm form) {
  constexpr int kPairs = 32 * GN * RN, kFeatures = 32 * GM * RM / (PRODUCT == kMoeGated ? 2 : 1);
  __shared__ u32x4 mem[WideShape<GM, GN, RM, RN>::kLds / 16];
  __shared__ int pairs[kPairs];  // of the tile; -1: beyond the list
  const int lane = threadIdx.x % kWave;
  const int features = (m + kFeatures - 1) / kFeatures;
  int total, e, within, row_tiles;
  moe_tile<kPairs>(counts, experts, n, features, -1, lane, total, e, within, row_tiles);
  total = __builtin_amdgcn_readfirstlane(total);
  const int die = blockIdx.x % 8, per_die = (total + 7) / 8, first = die * per_die;
  const int mine = min(per_die, total - first), whole = 2 * (mine % kDieRound) <= kDieRound ? mine / kDieRound * kDieRound : mine;
  int turn = blockIdx.x / 8, half = 0;
  const bool halved = turn >= whole;
  if (halved) half = (turn - whole) % 2, turn = whole + (turn - whole) / 2;
  if (turn >= mine) return;
  if (!moe_tile<kPairs>(counts, experts, n, features, first + turn, lane, total, e, within, row_tiles)) return;
  e = __builtin_amdgcn_readfirstlane(e);
  within = __builtin_amdgcn_readfirstlane(within);
  row_tiles = __builtin_amdgcn_readfirstlane(row_tiles);
  const int count = min(counts[e], n), row0 = within % row_tiles * kPairs;
  const int f0 = within / row_tiles * kFeatures + half * (kFeatures / 2);
  if (f0 >= m) return;
  const int32_t* list = order + static_cast<size_t>(e) * n;
  if (halved)
    moe_big_tile<PRODUCT, GM, GN, RM / 2, RN>(mem, pairs, e, f0, row0, count, a, list, w0, w1, act_out, pair_out, n, k, m, top, form);
  else
    moe_big_tile<PRODUCT, GM, GN, RM, RN>(mem, pairs, e, f0, row0, count, a, list, w0, w1, act_out, pair_out, n, k, m, top, form);
}

template <int PRODUCT, int GM, int GN, int RM, int RN>
static void launch_big(const bf16* a, const int32_t* order, const int32_t* counts, const void* w0, const void* w1, bf16* act_out,
                       float* pair_out, int n, int k, int m, int experts, int top, GateForm form, hipStream_t s) {
  constexpr int kPairs = 32 * GN * RN, kFeatures = 32 * GM * RM / (PRODUCT == kMoeGated ? 2 : 1);
  const long long features = (m + kFeatures - 1) / kFeatures, pairs = static_cast<long long>(n) * top;
  const long long tiles = features * (pairs / kPairs + (experts < pairs ? experts : pairs));  // live ones at most
  const long long groups = (tiles + 7) / 8 * 8 + 8 * (kDieRound / 2);  // (with the second halves of each die's last tiles)
  moe_big_mfma_kernel<PRODUCT, GM, GN, RM, RN><<<static_cast<unsigned>(groups), GM * GN * kWave, 0, s>>>(
      a, order, counts, static_cast<const bf16*>(w0), static_cast<const bf16*>(w1), act_out, pair_out, n, k, m, experts, top,
      form);
}

// A product per expert in the tile that wide_time() expects to be done first, as far as that can be known here: every
// list ends in half a tile, and `identity` of the router's outputs take their share of the pairs.  (Which tile makes no
// difference to the sums.)  A lane's values of the activation take 0.12 us each (measured while pieces left one by one; without
// that term both products of seven sizes at 400 to 8,192 tokens take 0.8 % less on average, but between 13 % less and 12 % more).  8 experts of
// 3584 x 4736, 1,501 tokens of two choices in 256 x 128, 256 x 192, 128 x 192, before tiles were halved: gate and up 231 / 228 / 237 us,
// down 143 / 103 / 123; 231 became 213.
constexpr int kBigTiles[] = {4, 1, 6};  // of kWide: 256 x 128, 256 x 192, 128 x 192
static int big_tile_of(int product, int n, int k, int m, int experts, int identity, int top) {
  const double pairs = static_cast<double>(n) * top * experts / (experts + identity);
  const int rows = product == kMoeGated ? 2 * m : m;
  int best = 0;
  double least = 0.0;
  for (int i = 0; i < 3; ++i) {
    WideTile t = kWide[kBigTiles[i]];
    if (product != kMoeDown) t.ends += 0.12 * (product == kMoeGated ? t.rows / 2 : t.rows) * t.tokens / (i ? 256 : 512);
    const double us = wide_time(t, ((rows + t.rows - 1) / t.rows) * (pairs / t.tokens + 0.5 * (experts < pairs ? experts : pairs)), k / 64);
    if (!i || us < least) least = us, best = i;
  }
  return best;
}

template <int PRODUCT>
static void big_product(const bf16* a, const int32_t* order, const int32_t* counts, const void* w0, const void* w1, bf16* act_out,
                        float* pair_out, int n, int k, int m, int experts, int identity, int top, GateForm form, hipStream_t s) {
  const int tile = big_tile_of(PRODUCT, n, k, m, experts, identity, top);
  const auto launch = tile == 0   ? launch_big<PRODUCT, 4, 2, 2, 2>
                      : tile == 1 ? launch_big<PRODUCT, 2, 2, 4, 3>
                                  : launch_big<PRODUCT, 2, 2, 2, 3>;
  launch(a, order, counts, w0, w1, act_out, pair_out, n, k, m, experts, top, form, s);
}

// Whether lists of 64 pairs and more keep moe_big_mfma_kernel's few, long workgroups busy for longer than they take to start and end,
// or the kernels for short lists, at about 200 TFLOP/s, are done before.  Both products and the join at 64 / 128 / 300 pairs a list, short lists'
// kernels against this one: 8 experts of 64 x 64 12 / 13 / 15 us against 22 / 24 / 26 (21 to 23 in the kernel for row-major
// weights), of 512 x 512 22 / 24 / 35 against 36 / 39 / 42, of 1024 x 1024 35 / 44 / 73 against 48 / 53 / 57, of 3584 x 1024
// 69 / 104 / 201 against 79 / 88 / 113; 32 of 512 x 512 35 / 51 / 92 against 40 / 46 / 69.  Up to 256 tokens the next power of two counts,
// so that a captured step decides as those it stands for.
// The short lists' grid has a place for every 32 tokens of each expert; those beyond a list's end, about 3,000 a microsecond, count too.
static bool fills_long_lists(int n, int top, int width, int ff, int experts, bool single) {
  long long tokens = n;
  for (int end = 32; end <= 256 && n <= 256; end *= 2)
    if (n <= end) {
      tokens = end;
      break;
    }
  const double flops = (single ? 4.0 : 6.0) * static_cast<double>(tokens * top) * width * ff;
  const double empty = top < experts ? (tokens + 31) / 32 * static_cast<double>(experts - top) * ((width + 31) / 32 + (ff + 31) / 32) : 0.0;
  return flops / 2e8 + empty / 3e3 >= 7.0 + 0.0125 * (width + ff);  // microseconds
}

// Tokens of one call with lists for moe_big_mfma_kernel, whose offsets within the tokens' rows, and within the pairs', are 32 bits
// wide; more of them are taken in several turns.
static int big_tokens(int n, int width, int ff, int top) {
  const long long row = width > static_cast<long long>(top) * ff ? width : static_cast<long long>(top) * ff;
  const long long most = ((1LL << 31) - 1) / row, turns = most ? (n + most - 1) / most : 1;
  return static_cast<int>((n + turns - 1) / turns);
}

// Which kernels take a step's products: 0 moe_big_mfma_kernel, 1 moe_tiled_mfma_kernel, 2 those for short lists.
static int experts_kernel(int n, int width, int ff, int experts, int top, bool single, bool tiled) {
  const bool many = static_cast<long long>(n) * top >= 64LL * experts;  // lists of 64 pairs and more on average
  if (many && !tiled) return 1;
  // (offsets within 256 rows of a matrix, and within a token's, are 32 bits wide)
  const bool near = width <= 1 << 22 && static_cast<long long>(top) * ff < 1LL << 31 && ff <= 1 << 22;
  return many && near && fills_long_lists(n, top, width, ff, experts, single) ? 0 : 2;
}

// out[t, c] = add[t, c] + sum_k weights[t, k] * pair_out[t * top + k, c], k in the order chosen; an identity
// expert's output is x[t, c].  Eight columns a thread (width is a multiple of 8): 16-byte loads and stores, 25 us
// at 1,501 tokens of 3584 with one column a thread, 13 so.  wide: add and out are 16-byte aligned,
// else element by element.  IDENTITY: a pair may be an identity expert's; the branch lets a token wait for each pair's output
// before it asks for the next (8 of 32 experts of 64 features, width 128, 8 tokens: all four launches 14.5 us, 12.1
// without).  From some 500 tokens on others cover that wait and the loop with the branch, which holds less in registers, is as fast
// or faster (128,000 tokens of one expert each, width 512: 780 us against 842).
template <bool IDENTITY>
__global__ void __launch_bounds__(256)
    moe_join_kernel(const float* __restrict__ pair_out, const int32_t* __restrict__ chosen, const bf16* __restrict__ x,
                    const float* __restrict__ weights, const bf16* __restrict__ add, const float* __restrict__ add_gate,
                    int gate_ld, bf16* __restrict__ out, int width, int top, int experts, int wide) {
  union Eight {
    uint4 u;
    bf16 h[8];
  };
  const int t = blockIdx.y;
  const int c = (blockIdx.x * blockDim.x + threadIdx.x) * 8;
  if (c >= width) return;
  const size_t at = static_cast<size_t>(t) * width + c;
  float total[8] = {};
  auto join = [&](int k) {
    const size_t pair = static_cast<size_t>(t) * top + k;
    const float weight = weights[pair];
    if (!IDENTITY || chosen[pair] < experts) {
      const float4 *y = reinterpret_cast<const float4*>(pair_out + pair * width + c);
      const float4 y0 = y[0], y1 = y[1];
      total[0] = fmaf(weight, y0.x, total[0]), total[1] = fmaf(weight, y0.y, total[1]);
      total[2] = fmaf(weight, y0.z, total[2]), total[3] = fmaf(weight, y0.w, total[3]);
      total[4] = fmaf(weight, y1.x, total[4]), total[5] = fmaf(weight, y1.y, total[5]);
      total[6] = fmaf(weight, y1.z, total[6]), total[7] = fmaf(weight, y1.w, total[7]);
    } else {
      Eight v;
      v.u = *reinterpret_cast<const uint4*>(x + at);
#pragma unroll
      for (int i = 0; i < 8; ++i) total[i] = fmaf(weight, to_float(v.h[i]), total[i]);
    }
  };
  if (IDENTITY) {
    for (int k = 0; k < top; ++k) join(k);
  } else {
#pragma unroll 4
    for (int k = 0; k < top; ++k) join(k);
  }
  if (add) {
    Eight v;
    if (wide)
      v.u = *reinterpret_cast<const uint4*>(add + at);
    else
#pragma unroll
      for (int i = 0; i < 8; ++i) v.h[i] = add[at + i];
    const float share = shared_share(add_gate, gate_ld, t);
#pragma unroll
    for (int i = 0; i < 8; ++i) total[i] += share * to_float(v.h[i]);
  }
  Eight v;
#pragma unroll
  for (int i = 0; i < 8; ++i) v.h[i] = from_float<bf16>(total[i]);
  if (wide)
    *reinterpret_cast<uint4*>(out + at) = v.u;
  else
#pragma unroll
    for (int i = 0; i < 8; ++i) out[at + i] = v.h[i];
}

}  // namespace shk

using namespace shk;

extern "C" int shk_moe_route(const float* logits, int ld, const float* correction, int experts, int top,
                             int groups, int keep, float scale, int32_t* chosen, float* weights, int n, void* stream) {
  SHK_REQUIRE(n >= 0 && experts > 0 && experts <= 8 * kWave && top >= 1 && top <= experts &&
                  top <= kWave && ld >= experts,
              "moe_route: bad sizes n=%d experts=%d top=%d", n, experts, top);
  SHK_REQUIRE(groups >= 1 && groups <= kWave && experts % groups == 0 && keep >= 1 && keep <= groups &&
                  top <= keep * (experts / groups),
              "moe_route: %d of %d experts cannot be chosen from %d of %d groups", top, experts, keep, groups);
  if (n == 0) return 0;
  SHK_REQUIRE(logits && chosen && weights, "moe_route: null pointer");
  const auto kernel = experts <= kWave ? moe_route_kernel<1> : moe_route_kernel<8>;
  kernel<<<(n + 3) / 4, 256, 0, static_cast<hipStream_t>(stream)>>>(logits, ld, correction, experts, top, groups, keep, scale, chosen,
                                                                    weights, n);
  SHK_LAUNCH_CHECK("moe_route");
  return 0;
}

extern "C" int shk_moe_experts(const void* x, const int32_t* chosen, const float* weights, const void* w_gate,
                               const void* w_up, const void* w_down, const void* add, const float* add_gate,
                               int gate_ld, void* act_buf, void* out, int dtype, int n, int width, int ff, int experts, int top,
                               int identity, int act, float limit, float shift, void* stream) {
  SHK_REQUIRE(dtype == kF32 || dtype == kBF16, "moe_experts: unknown dtype %d", dtype);
  SHK_REQUIRE(n >= 0 && width > 0 && ff > 0 && experts > 0 && identity >= 0 && top >= 1 && top <= experts + identity,
              "moe_experts: bad sizes n=%d width=%d ff=%d experts=%d top=%d", n, width, ff, experts, top);
  SHK_REQUIRE(act >= 1 && act <= 4, "moe_experts: unknown activation %d", act);
  SHK_REQUIRE(!add_gate || (add && gate_ld >= 1), "moe_experts: a gate of the added rows needs those rows and a stride");
  SHK_REQUIRE(width <= 15000 && static_cast<long long>(top) * ff <= 15000,
              "moe_experts: rows of %d, or %d chosen experts of %d features, do not fit a workgroup's LDS", width, top,
              ff);
  if (n == 0) return 0;
  SHK_REQUIRE(static_cast<long long>(n) * top <= 65535, "moe_experts: at most 65535 (token, expert) pairs a call");
  SHK_REQUIRE(x && chosen && weights && w_gate && w_up && w_down && act_buf && out, "moe_experts: null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const GateForm form{act, limit, shift};
  const dim3 g1((ff + kMoeFeatures - 1) / kMoeFeatures, n * top), g2((width + kMoeFeatures - 1) / kMoeFeatures, n);
#define SHK_GO(T)                                                                                                     \
  moe_gate_up_kernel<T><<<g1, 256, width * sizeof(float), s>>>(static_cast<const T*>(x), chosen,                      \
                                                               static_cast<const T*>(w_gate),                         \
                                                               static_cast<const T*>(w_up), static_cast<T*>(act_buf), \
                                                               width, ff, top, form, experts);                        \
  moe_down_kernel<T><<<g2, 256, static_cast<size_t>(top) * ff * sizeof(float), s>>>(                                  \
      static_cast<const T*>(x), static_cast<const T*>(act_buf), chosen, weights, static_cast<const T*>(w_down),       \
      static_cast<const T*>(add),                                                                                     \
      add_gate, gate_ld, static_cast<T*>(out), width, ff, top, experts)
  if (dtype == kF32) {
    SHK_GO(float);
  } else {
    SHK_GO(bf16);
  }
#undef SHK_GO
  SHK_LAUNCH_CHECK("moe_experts");
  return 0;
}

extern "C" long long shk_moe_grouped_scratch_bytes(int n, int width, int experts, int top) {
  // order [experts, n] and counts [experts] (int32), then the pairs' outputs [n * top, width] (float32)
  const long long ints = static_cast<long long>(experts) * n + experts;
  return ((ints * 4 + 15) / 16) * 16 + static_cast<long long>(n) * top * width * 4;
}

extern "C" int shk_moe_experts_plan(int n, int width, int ff, int experts, int top, int identity, int single, int tiled) {
  const int kernel = experts_kernel(n, width, ff, experts, top, single, tiled);
  if (kernel) return -kernel;
  n = big_tokens(n, width, ff, top);
  return 8 * kBigTiles[big_tile_of(single ? kMoeSingle : kMoeGated, n, width, ff, experts, identity, top)] +
         kBigTiles[big_tile_of(kMoeDown, n, ff, width, experts, identity, top)];
}

extern "C" int shk_moe_experts_grouped(const void* x, const int32_t* chosen, const float* weights, const void* w_gate,
                                       const void* w_up, const void* w_down, const void* add, const float* add_gate,
                                       int gate_ld, void* act_buf, void* out, void* scratch, int n, int width, int ff, int experts, int top,
                                       int identity, int act, float limit, float shift, int tiled, void* stream) {
  SHK_REQUIRE(n >= 0 && width > 0 && ff > 0 && experts > 0 && experts <= 65535 && identity >= 0 && top >= 1 && top <= experts + identity,
              "moe_experts_grouped: bad sizes n=%d width=%d ff=%d experts=%d top=%d", n, width, ff, experts, top);
  SHK_REQUIRE(act >= 1 && act <= 4, "moe_experts_grouped: unknown activation %d", act);
  SHK_REQUIRE(!add_gate || (add && gate_ld >= 1),
              "moe_experts_grouped: a gate of the added rows needs those rows and a stride");
  SHK_REQUIRE(width % 8 == 0 && ff % 8 == 0, "moe_experts_grouped: width %d and ff %d must be multiples of 8", width, ff);
  SHK_REQUIRE(!tiled || (width % 64 == 0 && ff % 64 == 0),
              "moe_experts_grouped: weights in tiles need a width %d and ff %d in multiples of 64", width, ff);
  if (n == 0) return 0;
  SHK_REQUIRE(static_cast<long long>(n) * top < (1LL << 30) && (n + 31) / 32 <= 65535,
              "moe_experts_grouped: too many (token, expert) pairs");
  SHK_REQUIRE(x && chosen && weights && w_gate && w_up && w_down && act_buf && out && scratch,
              "moe_experts_grouped: null pointer");
  for (const void* p : {x, w_gate, w_up, w_down, static_cast<const void*>(act_buf), static_cast<const void*>(scratch)})
    SHK_REQUIRE(reinterpret_cast<uintptr_t>(p) % 16 == 0, "moe_experts_grouped: operands must be 16-byte aligned");
  const int kernel = experts_kernel(n, width, ff, experts, top, w_gate == w_up, tiled);
  const int turn = kernel ? n : big_tokens(n, width, ff, top);
  if (turn < n) {
    for (int t = 0; t < n; t += turn) {
      const size_t at = t;
      const int failed = shk_moe_experts_grouped(
          static_cast<const bf16*>(x) + at * width, chosen + at * top, weights + at * top, w_gate, w_up, w_down,
          add ? static_cast<const bf16*>(add) + at * width : nullptr, add_gate ? add_gate + at * gate_ld : nullptr, gate_ld, act_buf,
          static_cast<bf16*>(out) + at * width, scratch, turn < n - t ? turn : n - t, width, ff, experts, top, identity, act, limit,
          shift, tiled, stream);
      if (failed) return failed;
    }
    return 0;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  const GateForm form{act, limit, shift};
  int32_t* order = static_cast<int32_t*>(scratch);
  int32_t* counts = order + static_cast<size_t>(experts) * n;
  const long long ints = static_cast<long long>(experts) * n + experts;
  float* pair_out = reinterpret_cast<float*>(static_cast<char*>(scratch) + ((ints * 4 + 15) / 16) * 16);
  moe_lists_kernel<<<experts, 256, 0, s>>>(chosen, n, top, order, counts);
  const bf16 *xb = static_cast<const bf16*>(x), *actb = static_cast<const bf16*>(act_buf);
  if (kernel == 0) {
    if (w_gate == w_up)
      big_product<kMoeSingle>(xb, order, counts, w_gate, w_up, static_cast<bf16*>(act_buf), nullptr, n, width, ff, experts, identity, top, form, s);
    else
      big_product<kMoeGated>(xb, order, counts, w_gate, w_up, static_cast<bf16*>(act_buf), nullptr, n, width, ff, experts, identity, top, form, s);
    big_product<kMoeDown>(actb, order, counts, w_down, nullptr, nullptr, pair_out, n, ff, width, experts, identity, top, form, s);
  } else if (kernel == 1) {
    const int row_tiles = (n + kTileRows - 1) / kTileRows;
    if (w_gate == w_up)
      moe_tiled_mfma_kernel<true, true><<<dim3((ff + 127) / 128, row_tiles, experts), 256, 0, s>>>(
          static_cast<const bf16*>(x), order, counts, static_cast<const bf16*>(w_gate), static_cast<const bf16*>(w_up),
          static_cast<bf16*>(act_buf), nullptr, n, width, ff, top, form);
    else
      moe_tiled_mfma_kernel<true><<<dim3((ff + 63) / 64, row_tiles, experts), 256, 0, s>>>(
          static_cast<const bf16*>(x), order, counts, static_cast<const bf16*>(w_gate), static_cast<const bf16*>(w_up),
          static_cast<bf16*>(act_buf), nullptr, n, width, ff, top, form);
    moe_tiled_mfma_kernel<false><<<dim3((width + 127) / 128, row_tiles, experts), 256, 0, s>>>(
        static_cast<const bf16*>(act_buf), order, counts, static_cast<const bf16*>(w_down), nullptr, nullptr, pair_out, n,
        ff, width, top, form);
  } else {
    const int row_tiles = (n + 31) / 32;
    const dim3 features((ff + 31) / 32, row_tiles, experts), columns((width + 31) / 32, row_tiles, experts);
    const bool single = w_gate == w_up;
    auto gate_up = tiled ? (single ? moe_gate_up_mfma_kernel<true, true> : moe_gate_up_mfma_kernel<false, true>)
                         : (single ? moe_gate_up_mfma_kernel<true, false> : moe_gate_up_mfma_kernel<false, false>);
    gate_up<<<features, 256, 0, s>>>(xb, order, counts, static_cast<const bf16*>(w_gate), static_cast<const bf16*>(w_up),
                                     static_cast<bf16*>(act_buf), n, width, ff, top, form);
    auto down = tiled ? moe_down_mfma_kernel<true> : moe_down_mfma_kernel<false>;
    down<<<columns, 256, 0, s>>>(actb, order, counts, static_cast<const bf16*>(w_down), pair_out, n, width, ff, top);
  }
  const int join_threads = width >= 2048 ? 256 : kWave;
  const int wide = reinterpret_cast<uintptr_t>(add) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
  auto join = identity || top == 1 || n > 512 ? moe_join_kernel<true> : moe_join_kernel<false>;
  join<<<dim3((width / 8 + join_threads - 1) / join_threads, n), join_threads, 0, s>>>(
      pair_out, chosen, xb, weights, static_cast<const bf16*>(add), add_gate, gate_ld, static_cast<bf16*>(out), width, top, experts, wide);
  SHK_LAUNCH_CHECK("moe_experts_grouped");
  return 0;
}
