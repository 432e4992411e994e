// The experts' products of up to 16 tokens (moe.hip says what they are), the shared expert's among them: a workgroup for a block of
// 16 weight rows of an expert that some token has chosen, formed as the few-token products of gemm_few.hip are.  Every workgroup lists
// its expert's pairs itself, and the shared expert is one more expert of the launch, which every token passes: its matrices stream
// beside the others' instead of behind them, and three kernels a layer are gone.
// What bounds it is the weights' stream.  Eight tokens, two of eight experts of 4736 over a width of 3584 beside a shared one of 9472: lists
// 4.6 us, experts 88 and 47, shared 26 and 23, join 4.8 in moe.hip's kernels for short lists and the plain products; a step of 28 such layers
// 7,570 us so, 6,490 here, one token 4,918 and 3,970, sixteen 8,615 and 7,246.
#include <cmath>

#include "gemm_few.h"

namespace shk {

struct MoeFewGate {
  int act;
  float limit, shift;
};

__device__ __forceinline__ float moe_few_gate(float g, float u, MoeFewGate form) {  // (as in moe.hip)
  if (form.limit > 0.f) {
    g = fminf(g, form.limit);
    u = fminf(fmaxf(u, -form.limit), form.limit);
  }
  u += form.shift;
  if (form.act == kActRelu) return fmaxf(g, 0.f) * u;
  const float x = form.act == kActGeluTanh ? 2.f * 0.7978845608028654f * (g + 0.044715f * g * g * g) : form.act == kActQuickGelu ? 1.702f * g : g;
  return g / (1.f + expf(-x)) * u;
}

constexpr int kMoeFewTop = 8;  // choices a token at most
// Wavefronts of a workgroup, which share k: the 7B sizes' step of eight sequences 6,490 us with 8 in both products, 6,566 with 4 in the
// second, 6,605 with 4 in the first.
constexpr int kMoeFewWaves = 8;

// The pairs (token * top + place among its choices) of expert e, tokens ascending: lane r < count holds the r-th.  The shared
// expert's r-th is token r.
struct MoeFewList {
  int count, mine;
  __device__ __forceinline__ MoeFewList(const int32_t* __restrict__ chosen, int n, int top, int e, bool shared, int* place) {
    const int lane = threadIdx.x % kWave;
    if (shared) {
      count = n, mine = lane;
      return;
    }
    int pick[kMoeFewTop];
    const int at = lane < n ? lane : n - 1;
#pragma unroll
    for (int k = 0; k < kMoeFewTop; ++k) pick[k] = chosen[at * top + (k < top ? k : 0)];
    int hit = -1;
#pragma unroll
    for (int k = kMoeFewTop - 1; k >= 0; --k)
      if (k < top && pick[k] == e) hit = k;
    const unsigned long long votes = __ballot(lane < n && hit >= 0);
    count = __popcll(votes);
    // the r-th hit's pair to lane r, through LDS of this wavefront's own; the fences order one lane's write and another's read
    if (lane < n && hit >= 0) place[__popcll(votes & ((1ull << lane) - 1ull))] = lane * top + hit;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    mine = place[lane < 16 ? lane : 0];
  }
};

struct MoeFewExperts {
  const int32_t* chosen;
  int n, top, experts;
};

// blockIdx.y: the expert; `experts` itself is the shared one (blocks of its gate and its other matrix lie in turn).
template <int WAVES>
__global__ void __launch_bounds__(WAVES* kWave)
    moe_few_gate_up_kernel(MoeFewExperts list, const bf16* __restrict__ x, int width, const u32x4* __restrict__ wg,
                           const u32x4* __restrict__ wu, int ff, MoeFewGate form, bf16* __restrict__ act_out,
                           const u32x4* __restrict__ shared, int shared_ff, MoeFewGate shared_form, bf16* __restrict__ shared_act) {
  __shared__ f32x4 red[WAVES][2][kWave];
  __shared__ int places[WAVES][16];
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int e = blockIdx.y, b = blockIdx.x, ktiles = width / 32;
  const bool all = e == list.experts;
  const int features = all ? shared_ff : ff;
  if (b * 16 >= features) return;
  const u32x4* gate = all ? shared + static_cast<size_t>(2 * b) * ktiles * kWave : wg + (static_cast<size_t>(e) * (ff / 16) + b) * ktiles * kWave;
  const u32x4* up = all ? gate + static_cast<size_t>(ktiles) * kWave : wu + (static_cast<size_t>(e) * (ff / 16) + b) * ktiles * kWave;
  const u32x4* const wrow[2] = {gate + lane, up + lane};
  const MoeFewList pairs(list.chosen, list.n, list.top, e, all, places[wave]);
  if (pairs.count == 0) return;
  f32x4 acc[2][1];
  few_multiply<0, 2, 2, 1>(
      acc, wrow,
      [&](const bf16* (&arow)[1]) {
        const int pair = __shfl(pairs.mine, min(lane % 16, pairs.count - 1), kWave);
        arow[0] = x + static_cast<size_t>(min(all ? pair : pair / list.top, list.n - 1)) * width;
      },
      1, width, ktiles, wave, WAVES, [] {});
  red[wave][0][lane] = acc[0][0];
  red[wave][1][lane] = acc[1][0];
  __syncthreads();
  for (int i = threadIdx.x; i < 256; i += WAVES * kWave) {
    const int inside = i / 16, r = i % 16;
    // (a lane's own list: 16 threads of a pair read it from the lane that holds it)
    const int pair = __shfl(pairs.mine, min(inside, pairs.count - 1), kWave);
    if (inside >= pairs.count) continue;
    const float g = few_sum(&red[0][0][0], 2 * kWave, r, inside, WAVES), u = few_sum(&red[0][1][0], 2 * kWave, r, inside, WAVES);
    bf16* row = all ? shared_act + static_cast<size_t>(pair) * shared_ff : act_out + static_cast<size_t>(pair) * ff;
    row[b * 16 + r] = from_float<bf16>(moe_few_gate(g, u, all ? shared_form : form));
  }
}

// pair_out[pair] = W_down_e . act[pair], shared_out[token] = W_down . shared_act[token]
template <int WAVES>
__global__ void __launch_bounds__(WAVES* kWave)
    moe_few_down_kernel(MoeFewExperts list, const bf16* __restrict__ act, int ff, const u32x4* __restrict__ wd, int width,
                        float* __restrict__ pair_out, const u32x4* __restrict__ shared, const bf16* __restrict__ shared_act,
                        int shared_ff, float* __restrict__ shared_out) {
  __shared__ f32x4 red[WAVES][kWave];
  __shared__ int places[WAVES][16];
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int e = blockIdx.y, b = blockIdx.x;
  const bool all = e == list.experts;
  const int k = all ? shared_ff : ff, ktiles = k / 32;
  const bf16* rows = all ? shared_act : act;
  const u32x4* const wrow[1] = {(all ? shared : wd + static_cast<size_t>(e) * (width / 16) * ktiles * kWave) +
                                static_cast<size_t>(b) * ktiles * kWave + lane};
  const MoeFewList pairs(list.chosen, list.n, list.top, e, all, places[wave]);
  if (pairs.count == 0) return;
  f32x4 acc[1][1];
  few_multiply<0, 4, 1, 1>(
      acc, wrow,
      [&](const bf16* (&arow)[1]) {
        const int pair = __shfl(pairs.mine, min(lane % 16, pairs.count - 1), kWave);
        arow[0] = rows + static_cast<size_t>(min(pair, list.n * (all ? 1 : list.top) - 1)) * k;
      },
      1, k, ktiles, wave, WAVES, [] {});
  red[wave][lane] = acc[0][0];
  __syncthreads();
  for (int i = threadIdx.x; i < 256; i += WAVES * kWave) {
    const int inside = i / 16, r = i % 16;
    const int pair = __shfl(pairs.mine, min(inside, pairs.count - 1), kWave);
    if (inside >= pairs.count) continue;
    (all ? shared_out : pair_out)[static_cast<size_t>(pair) * width + b * 16 + r] = few_sum(&red[0][0], kWave, r, inside, WAVES);
  }
}

// out[t] = sum over the choices, in order, of weight * pair_out (an identity expert: x[t] itself) + share * shared_out[t]
__global__ void __launch_bounds__(256)
    moe_few_join_kernel(MoeFewExperts list, const float* __restrict__ pair_out, const bf16* __restrict__ x, const float* __restrict__ weights,
                        const float* __restrict__ shared_out, const float* __restrict__ add_gate, int gate_ld, bf16* __restrict__ out,
                        int width) {
  const int t = blockIdx.y, c = (blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (c >= width) return;
  const size_t at = static_cast<size_t>(t) * width + c;
  const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 term[kMoeFewTop], total = zero, extra = zero;
  float weight[kMoeFewTop];
  const uint2 raw = *reinterpret_cast<const uint2*>(x + at);
  const f32x4 same = {__uint_as_float(raw.x << 16), __uint_as_float(raw.x & 0xffff0000u), __uint_as_float(raw.y << 16),
                      __uint_as_float(raw.y & 0xffff0000u)};
  if (shared_out) extra = *reinterpret_cast<const f32x4*>(shared_out + at);
  const float share = shared_out && add_gate ? 1.f / (1.f + expf(-add_gate[static_cast<size_t>(t) * gate_ld])) : 1.f;
#pragma unroll
  for (int k = 0; k < kMoeFewTop; ++k) {
    const int pair = t * list.top + (k < list.top ? k : 0);
    weight[k] = weights[pair];
    term[k] = same;
    if (list.chosen[pair] < list.experts) term[k] = *reinterpret_cast<const f32x4*>(pair_out + static_cast<size_t>(pair) * width + c);
  }
#pragma unroll
  for (int k = 0; k < kMoeFewTop; ++k)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (k < list.top) total[i] = fmaf(weight[k], term[k][i], total[i]);
  if (shared_out)
#pragma unroll
    for (int i = 0; i < 4; ++i) total[i] += share * extra[i];
  uint2 two;
  two.x = bf16_bits(total[0]) | static_cast<uint32_t>(bf16_bits(total[1])) << 16;
  two.y = bf16_bits(total[2]) | static_cast<uint32_t>(bf16_bits(total[3])) << 16;
  *reinterpret_cast<uint2*>(out + at) = two;
}

}  // namespace shk

using namespace shk;

extern "C" int shk_moe_few_takes(int n, int top) { return n <= 16 && top <= kMoeFewTop; }

// Whether a layer's steps of up to 16 tokens are faster here than in moe.hip's kernels for short lists and the shared expert's own products.
// What they save is one launch, with a shared expert four, and that weights stream side by side; what they cost is a workgroup for every block of
// every expert, chosen or not, and more of them than the other kernels where a block has pairs.  An estimate in microseconds, fitted to 1,755
// measured steps (2 to 512 experts of 64 x 64 to 7168 x 2048, shared ones of none to 9,472 features, 1 to 8 choices, 1 to 16 tokens): of the
// 755 that it takes, three are more than 2 % slower (up to 9), the others take 0.53 to 1.02 of the time.  Us at 1 / 4 / 16 tokens, there -> here, said
// to be faster: 8 experts of 3584 x 4736, two chosen, and a shared one of 9472 95 / 151 / 205 -> 76 / 124 / 165, of 896 x 1216 and 2432 25.3 / 28.2 / 32.1 ->
// 15.9 / 18.4 / 22.8, 16 of 512 x 512 and 512 18.8 / 19.4 / 20.7 -> 11.9 / 15.1 / 17.7, 8 of 64 x 64 alone 12.1 / 12.4 / 12.6 -> 9.5 / 9.9 / 10.6; not: 64 of 896 x
// 1216 and 2432 26.0 / 33.6 / 50.3 -> 27.6 / 35.1 / 54.9, 128 of 2048 x 768, eight chosen, 34.0 / 60.3 / 141 -> 49.2 / 87.6 / 180, 512 of them 41.5 / 68.0 / 191 ->
// 133 / 173 / 348, 16 of 512 x 512 alone 12.8 / 13.2 / 13.6 -> 12.0 / 14.4 / 15.9.  One answer for all numbers of tokens, which a recorded step stands for.
extern "C" int shk_moe_few_faster(int width, int ff, int shared_ff, int experts, int top, int identity) {
  if (experts < 1 || top < 1 || top > kMoeFewTop || top > experts + identity) return 0;
  const bool shared = shared_ff > 0;
  const double places = (experts + (shared ? 1 : 0)) * ((ff > shared_ff ? ff : shared_ff) + static_cast<double>(width)) / 16e3;
  for (int n : {1, 16}) {
    const double chosen = experts * (1.0 - std::pow(1.0 - static_cast<double>(top) / (experts + identity), n));
    const double blocks = chosen * (ff + static_cast<double>(width)) / 16e3, megabytes = 6e-6 * width * ff * chosen, beside = 6e-6 * width * shared_ff;
    if (2.0 + (shared ? 5.0 : 0.0) + 0.05 * megabytes + 0.11 * beside <= 0.9 * places + (4.0 + 0.07 * n) * blocks) return 0;
  }
  return 1;
}

extern "C" int shk_moe_few(const void* x, const int32_t* chosen, const float* weights, const void* w_gate, const void* w_up,
                           const void* w_down, const void* shared_gate_up, const void* shared_down, const float* add_gate, int gate_ld,
                           void* act_buf, void* shared_act, float* pair_out, void* out, int n, int width, int ff, int shared_ff,
                           int experts, int top, int identity, int act, float limit, float shift, float shared_limit, void* stream) {
  SHK_REQUIRE(n >= 0 && n <= 16 && width > 0 && width % 64 == 0 && ff > 0 && ff % 64 == 0 && experts > 0 && experts < 65535 && identity >= 0 &&
                  top >= 1 && top <= kMoeFewTop && top <= experts + identity,
              "moe_few: bad sizes n=%d width=%d ff=%d experts=%d top=%d", n, width, ff, experts, top);
  SHK_REQUIRE(act >= 1 && act <= kActQuickGelu && limit >= 0.f && shared_limit >= 0.f, "moe_few: unknown gate");
  SHK_REQUIRE((shared_gate_up != nullptr) == (shared_ff > 0) && shared_ff % 32 == 0, "moe_few: a shared expert of %d features", shared_ff);
  if (n == 0) return 0;
  SHK_REQUIRE(x && chosen && weights && w_gate && w_up && w_down && act_buf && pair_out && out && (!shared_gate_up || (shared_down && shared_act)),
              "moe_few: null pointer");
  for (const void* p : {x, w_gate, w_up, w_down, shared_gate_up, shared_down, static_cast<const void*>(act_buf),
                        static_cast<const void*>(shared_act), static_cast<const void*>(pair_out), static_cast<const void*>(out)})
    SHK_REQUIRE(reinterpret_cast<uintptr_t>(p) % 16 == 0, "moe_few: operands must be 16-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const MoeFewExperts list = {chosen, n, top, experts};
  const int lists = experts + (shared_gate_up ? 1 : 0);
  float* shared_out = shared_gate_up ? pair_out + static_cast<size_t>(n) * top * width : nullptr;
  const dim3 features(((ff > shared_ff ? ff : shared_ff) + 15) / 16, lists);
  moe_few_gate_up_kernel<kMoeFewWaves><<<features, kMoeFewWaves * kWave, 0, s>>>(
      list, static_cast<const bf16*>(x), width, static_cast<const u32x4*>(w_gate), static_cast<const u32x4*>(w_up), ff,
      MoeFewGate{act, limit, shift}, static_cast<bf16*>(act_buf), static_cast<const u32x4*>(shared_gate_up), shared_ff,
      MoeFewGate{act, shared_limit, shift}, static_cast<bf16*>(shared_act));
  moe_few_down_kernel<kMoeFewWaves><<<dim3(width / 16, lists), kMoeFewWaves * kWave, 0, s>>>(
      list, static_cast<const bf16*>(act_buf), ff, static_cast<const u32x4*>(w_down), width, pair_out,
      static_cast<const u32x4*>(shared_down), static_cast<const bf16*>(shared_act), shared_ff, shared_out);
  moe_few_join_kernel<<<dim3((width / 4 + 255) / 256, n), 256, 0, s>>>(list, pair_out, static_cast<const bf16*>(x), weights, shared_out,
                                                                      add_gate, gate_ld, static_cast<bf16*>(out), width);
  SHK_LAUNCH_CHECK("moe_few");
  return 0;
}
