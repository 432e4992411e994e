// The loop of products whose operands go from global memory straight into LDS, for the kernels that wrap it
// (gemm_wide.hip, moe.hip).
//
// A workgroup of GM x GN wavefronts forms 32*GM*RM weight rows x 32*GN*RN tokens, each wavefront RM x RN tiles of 32 x 32
// (v_mfma_f32_32x32x16_bf16: half the operand reads of the 16 x 16 form for the same product, and the same sums).
// Weights come in tiles of 16 rows x 32 of k (1 KiB, lane l of a wavefront holding row l % 16, k (l / 16) * 8 .. + 8).
//
// k is walked in substeps of 32 (a weight tile) and stages of 64 (whole cache lines of activations).  Weights live in a
// ring of four substeps, activations in a ring of three stages, so that what is loaded has three substeps to arrive.
// A wavefront multiplies half a substep (16 of k) while it reads the operands of the next half from LDS: one read behind
// each of the first multiplications, then the loads that refill what the barrier has just freed.  The barrier stands
// in the middle of a substep, where all its operands have been read.
//
// What bounds it: where every compute unit works, the power limit.  A stage of the 256 x 256 tile takes 2,180 cycles, the
// multiplications alone 2,048 to 2,110, at 1.55 to 1.6 GHz.  A load of activations takes 8 tokens x 128 bytes:
// neighbouring lanes on one token's line cost what a contiguous load costs, a lane a token 20 % of the loop (2,634
// cycles a stage).  The pieces of a line are stored rotated by token (piece c at place c ^ (token % 8)), so that the
// reads of the operands, 32 tokens at one piece, meet no bank conflicts.  Rings of six and eight substeps for the smaller
// tiles, and loads spread over the half instead of right behind the barrier, were as fast.
#pragma once

#include "common.h"
#include "to_lds.h"

namespace shk {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

template <int GM, int GN, int RM, int RN>
struct WideShape {
  static constexpr int kWaves = GM * GN;
  static constexpr int kTiles = 2 * GM * RM, kUnits = 4 * GN * RN;      // KiB of a substep's weights, of a stage's activations
  static constexpr int kWLoads = kTiles / kWaves, kXLoads = kUnits / kWaves / 2;  // of a wavefront, a substep
  static constexpr int kDepth = 3, kWRing = kDepth + 1, kXRing = kDepth;          // substeps; substeps; stages
  static constexpr int kWBytes = kTiles * 1024, kXBytes = kUnits * 1024;
  static constexpr int kLds = kWRing * kWBytes + kXRing * kXBytes;
  static_assert(kWLoads * kWaves == kTiles && 2 * kXLoads * kWaves == kUnits, "loads divide evenly among the wavefronts");
  // (a load stands behind each of a half's multiplications or reads but the first)
  static_assert(kWLoads < (RM * RN > RM + RN ? RM * RN : RM + RN) && kXLoads < (RM * RN > RM + RN ? RM * RN : RM + RN),
                "a half substep has a place for each of its loads");
  static_assert(kLds <= 160 * 1024 && kDepth * (kWLoads + kXLoads) <= 63, "fits LDS and the load counter");
  static_assert(kWaves * 32 * (32 * RM * 4 + 16) <= kLds, "the results of 32 tokens a wavefront fit LDS");
};


// acc = the product.  mem: S::kLds bytes of LDS.  wsrc + woff[i]: this lane's 16 bytes of weight tile wave + kWaves * i
// of the first substep, a substep 1,024 bytes.  xsrc + xoff[i]: its 16 bytes of unit wave + kWaves * i (8 tokens) of the
// first stage, piece (lane % 8) ^ (lane / 8) of token lane / 8, a stage 128 bytes.  In stage `last` (-1: none) `beyond`
// is taken off xoff: 16 * piece for a piece beyond k, the stage's first then standing in (numbers that meet the zeros which
// pad the weight tiles).  subs: substeps, stages: (subs + 1) / 2, at least one.  When it returns nothing is
// loaded into LDS or read from it any more.
template <int GM, int GN, int RM, int RN>
__device__ __forceinline__ void wide_loop(f32x16 (&acc)[RM][RN], u32x4* mem, const char* wsrc,
                                          const unsigned (&woff)[WideShape<GM, GN, RM, RN>::kWLoads], const char* xsrc,
                                          const unsigned (&xoff)[2 * WideShape<GM, GN, RM, RN>::kXLoads], unsigned beyond, int last,
                                          int subs, int stages) {
  using S = WideShape<GM, GN, RM, RN>;
  constexpr int N = RM * RN, R = RM + RN, WL = S::kWLoads, XL = S::kXLoads;
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int wm = wave / GN, wn = wave % GN;
  const unsigned base = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)mem)) + wave * 1024;
  constexpr int kX0 = S::kWRing * S::kWBytes;  // where the activations' ring begins

  // (past the share's end: substep or stage 0 again, never multiplied)
  auto load_w = [&](int at, int sub, int i) {
    SHK_LOAD_TO_LDS(base + at + i * S::kWaves * 1024, woff[i], wsrc + static_cast<size_t>(sub < subs ? sub : 0) * 1024);
  };
  auto load_x = [&](int at, int st, int half, int i) {
    st = st < stages ? st : 0;
    const unsigned cut = st == last ? ~0u : 0u;
    SHK_LOAD_TO_LDS(base + kX0 + at + (half * XL + i) * S::kWaves * 1024, xoff[half * XL + i] - (beyond & cut),
                    xsrc + static_cast<size_t>(st) * 128);
  };

#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int jn = 0; jn < RN; ++jn)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][jn][r] = 0.f;

  // Operands of 16 of k: lane l holds row (or token) l % 32, k (l / 32) * 8 .. + 8 of them.
  const char* lds = reinterpret_cast<const char*>(mem);
  const int wat = (wm * RM * 2 + (lane % 32) / 16) * 1024 + ((lane / 32) * 16 + lane % 16) * 16;
  int xat[4];
#pragma unroll
  for (int c = 0; c < 4; ++c)
    xat[c] = kX0 + (wn * RN * 32 + lane % 32) * 128 + ((2 * c + lane / 32) ^ (lane % 8)) * 16;
  struct Operands {
    u32x4 w[RM], x[RN];
  } even, odd;
  // operand i of half h of a substep in the weights' ring at `watp`, the stage's substep p in the activations' at `xatp`
  auto read = [&](Operands& f, int watp, int xatp, int p, int h, int i) {
    if (i < RM)
      f.w[i] = *reinterpret_cast<const u32x4*>(lds + wat + watp + i * 2048 + 512 * h);
    else
      f.x[i - RM] = *reinterpret_cast<const u32x4*>(lds + xat[2 * p + h] + xatp + (i - RM) * 4096);
  };
  auto multiply = [&](const Operands& f, int q) {
    const int i = q / RN, jn = q % RN;
    acc[i][jn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, f.w[i]),
                                                         __builtin_bit_cast(bf16x8, f.x[jn]), acc[i][jn], 0, 0, 0);
  };
  auto after_w = [](int at, int by) {
    return at + by * S::kWBytes < S::kWRing * S::kWBytes ? at + by * S::kWBytes : at + (by - S::kWRing) * S::kWBytes;
  };
  auto after_x = [](int at, int by) {
    return at + by * S::kXBytes < S::kXRing * S::kXBytes ? at + by * S::kXBytes : at + (by - S::kXRing) * S::kXBytes;
  };

  // Loads go out in the order in which they are waited for: per substep its weights and half a stage of activations.
#pragma unroll
  for (int i = 0; i < XL; ++i) load_x(0, 0, 0, i);
#pragma unroll
  for (int sub = 0; sub < S::kWRing; ++sub) {
#pragma unroll
    for (int i = 0; i < WL; ++i) load_w(sub * S::kWBytes, sub, i);
#pragma unroll
    for (int i = 0; i < XL; ++i) load_x((sub + 1) / 2 * S::kXBytes, (sub + 1) / 2, (sub + 1) % 2, i);
  }
  SHK_MEET_WITH_LOADS(S::kDepth * (WL + XL));
#pragma unroll
  for (int i = 0; i < R; ++i) read(even, 0, 0, 0, 0, i);
// Half a substep: its multiplications, and behind each of the first a read for the next half and one of the loads.
// Nothing is moved across sched_barrier, so this is the order in which they are issued.
#define SHK_WIDE_HALF(now, next, watp, xatp, p, h, loads, LOAD) \
  _Pragma("unroll") for (int q = 0; q < (N > R ? N : R); ++q) { \
    if (q < N) multiply(now, q);                                \
    if (q < R) read(next, watp, xatp, p, h, q);                 \
    if (q >= 1 && q <= loads) {                                 \
      const int i = q - 1;                                      \
      LOAD;                                                     \
    }                                                           \
    __builtin_amdgcn_sched_barrier(0);                          \
  }
// The stage's first substep from its second half on, its second substep's first half.
#define SHK_WIDE_STAGE()                                                             \
  SHK_MEET_WITH_LOADS((S::kDepth - 1) * (WL + XL));                                  \
  const int w1 = after_w(wp, 1), xlast = after_x(xp, S::kXRing - 1);                 \
  SHK_WIDE_HALF(odd, even, w1, xp, 1, 0, WL, load_w(wp, 2 * s + S::kWRing, i))       \
  SHK_WIDE_HALF(even, odd, w1, xp, 1, 1, XL, load_x(xlast, s + S::kXRing - 1, 1, i))
  int s = 0, wp = 0, xp = 0;  // stage; where its first substep and its activations lie in the rings
  SHK_WIDE_HALF(even, odd, 0, 0, 0, 1, 0, (void)i)
  for (; s + 1 < stages; ++s) {
    SHK_WIDE_STAGE()
    SHK_MEET_WITH_LOADS((S::kDepth - 1) * (WL + XL));
    const int w2 = after_w(wp, 2), x1 = after_x(xp, 1);
    SHK_WIDE_HALF(odd, even, w2, x1, 0, 0, WL, load_w(w1, 2 * s + 1 + S::kWRing, i))
    SHK_WIDE_HALF(even, odd, w2, x1, 0, 1, XL, load_x(xp, s + S::kXRing, 0, i))
    wp = w2, xp = x1;
  }
  if (2 * s + 1 < subs) {
    SHK_WIDE_STAGE()
  }
#pragma unroll
  for (int q = 0; q < N; ++q) multiply(odd, q);
#undef SHK_WIDE_HALF
#undef SHK_WIDE_STAGE
  SHK_WAIT_LOADS(0);
  __syncthreads();
}

// The tiles, and what they were measured to take: a workgroup's start and end, a stage of 64 of k with the chip nearly
// empty (its loads' latency) and what is added when all its compute units work (the power limit), in us; workgroups that
// fit on the chip.  From 13 products of 512 to 8,192 tokens in one to three shares: within 15 % of nearly all.  Over 2,568 of 100 to
// 4,000 tokens, 384 to 5,120 rows and up to eleven shares, weights in cache, 0.71 to 1.29 of the time in nine of ten.  (Both while tiles were dealt
// out in another order, see tile_of: products of few shares and many tokens then took up to half as long again.)
struct WideTile {
  int rows, tokens, units;
  double ends, alone, full;
};
constexpr WideTile kWide[] = {{256, 256, 256, 5.0, 0.897, 0.663}, {256, 192, 256, 7.0, 0.720, 0.460}, {192, 256, 256, 7.0, 0.791, 0.400},
                                 {192, 192, 256, 7.0, 0.524, 0.405}, {256, 128, 256, 3.5, 0.718, 0.167}, {128, 256, 256, 5.0, 0.631, 0.205},
                                 {128, 192, 256, 5.0, 0.428, 0.224}, {128, 128, 512, 3.5, 0.360, 0.620}};
constexpr int kWideTiles = sizeof(kWide) / sizeof(kWide[0]);

// Microseconds of `groups` workgroups of a tile, each walking `stages` stages of k.
inline double wide_time(const WideTile& t, double groups, int stages) {
  const double rounds = static_cast<double>(static_cast<long long>(groups) / t.units);
  double rest = (groups - rounds * t.units) / t.units;
  // (two on some compute units take as long as two on all: 296 of 128 x 128 x 3584 at 128 tokens 78 us, 148 of 256 x 128 66)
  if (t.units > 256 && rest > 0.5) rest = 1.0;
  double us = 2.0 + rounds * (t.ends + stages * (t.alone + t.full));
  if (rest > 0.0) us += t.ends + stages * (t.alone + t.full * rest);
  return us;
}

// Until this wavefront's accesses to LDS are done.
#define SHK_LDS_DONE() asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory")

}  // namespace shk
