// Causal grouped-query attention over the paged cache in float32 on the matrix units
// (v_mfma_f32_16x16x4_f32): one workgroup of four wavefronts per (token, key/value head, 16 of its
// query heads), the heads being the columns of both products, S^T = K Q^T and O^T = V^T P^T.
//
// A float32 result has the same bits however a prompt is cut, so the order of every sum follows from
// the key's position alone: keys are taken in blocks of 256 counted from position 0, a wavefront has
// the same 64 of each; a block has a maximum and sums of its own (the wavefronts' in order), and the
// blocks are joined in order with a running maximum.  A masked key has weight 0 and values that are
// read as 0 (its slot may hold anything), which changes no sum, so nothing depends on where a window
// begins within a block.  Single tokens may have their blocks formed by workgroups of their own
// (kSplit), whose results attention_f32_join_kernel joins by the same arithmetic.
//
// A lane of the first product's result holds four neighbouring keys of one head, which is the second
// product's operand as it stands: weights never pass through LDS.  What bounds it: a block is 64 + 64
// instructions of 32 cycles per wavefront (head size 64: 4,096 cycles) and three barriers.  14 heads of 64
// over 2, 509 tokens: 560 us a layer in the general kernel, whose one workgroup per query head had one key
// per thread, 38 with a workgroup a token, 24 with one for two (kPair: most of the 16 columns then hold a head); four single tokens at about 400: 50 us, here 12 and 4.4 for the join (whole passes: a
// prompt of 24 such layers 18.9 ms then, 6.5 with a workgroup a token; a decode step of four requests 2.43 ms, 1.56 now).  A
// single token's block is one chain from the page numbers over keys and values to the join, so all page
// numbers are read first, without a branch, then as many steps' keys and values as registers hold before the
// first product (head size 64: all of them; with each step's loads next to its products 16 us for the 12).  A
// prompt's tokens, with workgroups enough to cover one another's waits, take 6.5 ms either way.
#include "api.h"
#include "attention_f32.h"
#include "common.h"

namespace shk {

typedef float af4 __attribute__((ext_vector_type(4)));

constexpr int kBlockWaves = 4, kWaveKeys = kKeyBlock / kBlockWaves;

// (m, l) joins (M, L); e0 and e1 are the factors of what has been summed and of what joins.
__device__ __forceinline__ void join_block(float& M, float& L, float m, float l, float& e0, float& e1) {
  const float top = fmaxf(M, m);
  e0 = M == -INFINITY ? 0.f : expf(M - top);
  e1 = m == -INFINITY ? 0.f : expf(m - top);
  L = __fmaf_rn(L, e0, __fmul_rn(l, e1));
  M = top;
}

__device__ __forceinline__ float joined(float sum, float e0, float block, float e1) {
  return __fmaf_rn(sum, e0, __fmul_rn(block, e1));
}

// the sink joins the denominator alone
__device__ __forceinline__ float keys_share(float M, float& L, const float* sinks, int head) {
  if (!sinks) return 1.f;
  const float sink = sinks[head], top = fmaxf(M, sink), share = expf(M - top);
  L = L * share + expf(sink - top);
  return share;
}

// D: sixteens of the larger of head_dim and v_dim.  kPair: up to eight query heads a key/value head, whose columns two
// neighbouring tokens of one sequence share, the first in columns 0 to 7.
template <int D, bool kSplit, bool kPair>
__global__ void __launch_bounds__(kWave * kBlockWaves) attention_f32_kernel(F32Attention p, int n) {
  __shared__ af4 sums[kBlockWaves][D][kWave];
  __shared__ float tops[kBlockWaves][16], weights[kBlockWaves][16];
  const int lane = threadIdx.x % kWave, i = lane % 16, kg = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int per = p.heads / p.kv_heads, parts = (per + 15) / 16;
  const int kvh = blockIdx.x / parts, in_group = kPair ? i % 8 : blockIdx.x % parts * 16 + i;
  // (pairs first, the last of the prompt's before the others, then the tokens that most often are a pair's second: in the order
  // of the tokens every other workgroup would have nothing to do, and with two key/value heads so would four of the eight dies)
  const int pairs = (n + 1) / 2, y = blockIdx.y;
  const int t0 = !kPair ? y : y < pairs ? 2 * (pairs - 1 - y) : 2 * (y - pairs) + 1, seq = p.token_seq[t0];
  const int pos0 = p.positions[t0];
  int t1 = t0, pos1 = pos0;  // the token of columns 8 to 15
  if constexpr (kPair) {
    // (the other token of a pair; read without a condition, so that these loads travel together)
    const int other = min(t0 ^ 1, n - 1), beside = p.positions[other];
    const bool same = other != t0 && p.token_seq[other] == seq;
    if (same && t0 % 2) return;
    if (same) t1 = other, pos1 = beside;
  }
  const int lo0 = first_key(pos0, p.window, p.chunk), lo1 = kPair ? first_key(pos1, p.window, p.chunk) : lo0;
  const bool later = kPair && i >= 8;  // this column's token is t1
  const int t = later ? t1 : t0;
  const bool row = in_group < per && (!later || t1 != t0);
  const int head = kvh * per + (kPair ? min(in_group, per - 1) : row ? in_group : 0);
  // keys of either token, of this column's
  const int pos = kPair ? max(pos0, pos1) : pos0, lo = kPair ? min(lo0, lo1) : lo0;
  const int mine_to = later ? pos1 : pos0, mine_from = later ? lo1 : lo0;
  const int32_t* table = p.tables + static_cast<size_t>(seq) * p.table_stride;
  int first = lo / kKeyBlock, last = pos / kKeyBlock, step = 1;
  if (kSplit) {
    first += blockIdx.z;
    step = gridDim.z;
    if (first > last) return;
  }

  const float* qr = p.q + static_cast<size_t>(t) * p.q_stride + head * p.head_dim;
  af4 qv[D];
#pragma unroll
  for (int s = 0; s < D; ++s)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int d = 16 * s + 4 * kg + e;
      const float x = qr[d < p.head_dim ? d : 0];
      qv[s][e] = row && d < p.head_dim ? x : 0.f;
    }

  constexpr int kOwn = (D + kBlockWaves - 1) / kBlockWaves;  // tiles of values that this wavefront joins: wave, wave + 4, ..
  af4 own[kOwn];
#pragma unroll
  for (int o = 0; o < kOwn; ++o) own[o] = af4{0.f, 0.f, 0.f, 0.f};
  float M = -INFINITY, L = 0.f;
  const int slab = key_slab(p.head_dim), ps = p.page_size;
  const size_t k_page = static_cast<size_t>(ps) * p.head_dim, v_page = static_cast<size_t>(ps) * p.v_dim;
  // steps of 16 keys, how many are loaded at once, and how many are multiplied side by side
  constexpr int kSteps = kWaveKeys / 16, kAhead = D <= 4 ? kSteps : D <= 8 ? 2 : 1, kGroup = D <= 3 ? 2 : kAhead;
  auto page_of = [&](int key) {  // of `key`, or of the nearest key that is read; -1 where there is none
    const int page = table[min(max(key, lo), pos) / ps];
    return page < p.num_pages ? page : -1;
  };

  for (int b = first; b <= last; b += step) {
    const int key0 = b * kKeyBlock + wave * kWaveKeys;
    const bool any = key0 <= pos && key0 + kWaveKeys > lo;  // of this wavefront's keys is read
    // whether a group of steps holds a key that is read, for heads of up to 48 and of more than 128 (a prompt of 17 tokens,
    // heads of 32 7.2 us with all products, 6.4 so, of 256 27 and 20).  Those between lose more by the branch
    // than they gain (64: 500 tokens 37.6 us, 38.5 with it; 128: a second workgroup no longer fits on a compute
    // unit) and take up to 0.6 (64) and 1.9 us (16 heads of 128) longer than the general kernel for 17 tokens
    auto read = [&](int u) { return (D > 3 && D <= 8) || (key0 + 16 * u <= pos && key0 + 16 * (u + kGroup) > lo); };
    // scores: this lane loads key key0 + 16 u + i, and gets keys key0 + 16 u + 4 kg + 0..3 of head i
    af4 s[kSteps];
    int k_at[kSteps], v_at[kSteps];  // pages of the keys, and of the values, that this lane loads
    af4 kv[kAhead][D], vv[kAhead][D];
    auto load_keys = [&](int u) {
      const int key = key0 + 16 * u + i;
      const float* kr = p.k_pool + (static_cast<size_t>(max(k_at[u], 0)) * p.kv_heads + kvh) * k_page + static_cast<size_t>(key % ps) * slab;
#pragma unroll
      for (int x = 0; x < D; ++x) {
        const int d = 16 * x + 4 * kg;
        const size_t at = d < p.head_dim ? static_cast<size_t>(d / slab) * ps * slab + d % slab : 0;
        kv[u % kAhead][x] = *reinterpret_cast<const af4*>(kr + at);
      }
    };
    auto load_values = [&](int u) {
      const int key = key0 + 16 * u + 4 * kg;
      const float* vr = p.v_pool + (static_cast<size_t>(max(v_at[u], 0)) * p.kv_heads + kvh) * v_page + key % ps;
#pragma unroll
      for (int x = 0; x < D; ++x) {
        const int d = 16 * x + i;
        vv[u % kAhead][x] = *reinterpret_cast<const af4*>(vr + static_cast<size_t>(d < p.v_dim ? d : 0) * ps);
      }
    };
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
      s[u] = af4{0.f, 0.f, 0.f, 0.f};
      v_at[u] = -1;
    }
    if (any) {
#pragma unroll
      for (int u = 0; u < kSteps; ++u) {
        // (page sizes are multiples of four: a lane's four keys share a page, and where any of them is read
        // the nearest to the first that is read is one of them)
        k_at[u] = page_of(key0 + 16 * u + i);
        v_at[u] = page_of(key0 + 16 * u + 4 * kg);
      }
#pragma unroll
      for (int u0 = 0; u0 < kSteps; u0 += kAhead) {
        const bool loads = D <= 4 || read(u0);
        if (loads)
#pragma unroll
          for (int u = u0; u < u0 + kAhead; ++u) load_keys(u);
        if (u0 + kAhead == kSteps)
#pragma unroll
          for (int u = 0; u < kAhead; ++u) load_values(u);
#pragma unroll
        for (int g = u0; g < u0 + kAhead; g += kGroup) {
          if (!read(g)) continue;
#pragma unroll
          for (int x = 0; x < D; ++x)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
              for (int u = g; u < g + kGroup; ++u) {
                const float key = 16 * x + 4 * kg < p.head_dim ? kv[u % kAhead][x][e] : 0.f;
                s[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(key, qv[x][e], s[u], 0, 0, 0);
              }
        }
      }
    }
    float top = -INFINITY;
#pragma unroll
    for (int u = 0; u < kSteps; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int key = key0 + 16 * u + 4 * kg + e;
        float x = s[u][e] * p.scale;
        if (p.softcap > 0.f) x = p.softcap * tanhf(x / p.softcap);
        const bool have = key >= mine_from && key <= mine_to && v_at[u] >= 0;
        if (p.dist_bias && have) x += p.dist_bias[static_cast<size_t>(head) * p.bias_rows + min(mine_to - key, p.bias_rows - 1)];
        s[u][e] = have ? x : -INFINITY;
        top = fmaxf(top, s[u][e]);
      }
    top = fmaxf(top, __shfl_xor(top, 16));
    top = fmaxf(top, __shfl_xor(top, 32));
    if (kg == 0) tops[wave][i] = top;
    __syncthreads();
    float m = tops[0][i];
#pragma unroll
    for (int w = 1; w < kBlockWaves; ++w) m = fmaxf(m, tops[w][i]);
    // (scores may be -infinity by themselves, from a table of distances or an overflow: a block of them has weights of 0)
    const float origin = m == -INFINITY ? 0.f : m;

    float l = 0.f;
    af4 acc[D];
#pragma unroll
    for (int x = 0; x < D; ++x) acc[x] = af4{0.f, 0.f, 0.f, 0.f};
    if (any) {
#pragma unroll
      for (int u = 0; u < kSteps; ++u) {
        if (!read(u / kGroup * kGroup)) continue;
        if (u >= kAhead && u % kAhead == 0)
#pragma unroll
          for (int ahead = u; ahead < u + kAhead; ++ahead) load_values(ahead);
        // what one of two tokens may read and the other may not must not meet the other's weight of 0 (it may be infinite)
        const int step0 = key0 + 16 * u;
        if (kPair && ((pos0 != pos1 && step0 <= pos && step0 + 15 > min(pos0, pos1)) ||
                      (lo0 != lo1 && step0 < max(lo0, lo1) && step0 + 15 >= lo))) {
          af4 other[D];
#pragma unroll
          for (int x = 0; x < D; ++x) other[x] = acc[x];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int key = step0 + 4 * kg + e;
            const bool have0 = key >= lo0 && key <= pos0 && v_at[u] >= 0, have1 = key >= lo1 && key <= pos1 && v_at[u] >= 0;
            const float w = (i < 8 ? have0 : have1) ? expf(s[u][e] - origin) : 0.f;
            l += w;
#pragma unroll
            for (int x = 0; x < D; ++x) {
              acc[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(have0 ? vv[u % kAhead][x][e] : 0.f, w, acc[x], 0, 0, 0);
              other[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(have1 ? vv[u % kAhead][x][e] : 0.f, w, other[x], 0, 0, 0);
            }
          }
#pragma unroll
          for (int x = 0; x < D; ++x)
            if (i >= 8) acc[x] = other[x];
          continue;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int key = key0 + 16 * u + 4 * kg + e;
          const bool have = key >= lo && key <= pos && v_at[u] >= 0;
          const float w = have ? expf(s[u][e] - origin) : 0.f;
          l += w;
#pragma unroll
          for (int x = 0; x < D; ++x)
            acc[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(have ? vv[u % kAhead][x][e] : 0.f, w, acc[x], 0, 0, 0);
        }
      }
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (kg == 0) weights[wave][i] = l;
#pragma unroll
    for (int x = 0; x < D; ++x) sums[wave][x][lane] = acc[x];
    __syncthreads();
    l = weights[0][i];
#pragma unroll
    for (int w = 1; w < kBlockWaves; ++w) l += weights[w][i];
    float e0 = 0.f, e1 = 1.f;
    if (!kSplit) join_block(M, L, m, l, e0, e1);
    float* mine = kSplit ? p.partial + ((static_cast<size_t>(t) * p.heads + head) * p.blocks + b) * (p.v_dim + 2) : nullptr;
    if (kSplit && row && wave == 0 && kg == 0) {
      mine[p.v_dim] = m;
      mine[p.v_dim + 1] = l;
    }
#pragma unroll
    for (int o = 0; o < kOwn; ++o) {
      const int x = wave + o * kBlockWaves;
      if (x >= D) continue;
      af4 v = sums[0][x][lane];
#pragma unroll
      for (int w = 1; w < kBlockWaves; ++w) v += sums[w][x][lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int d = 16 * x + 4 * kg + e;
        if (!kSplit)
          own[o][e] = joined(own[o][e], e0, v[e], e1);
        else if (row && d < p.v_dim)
          mine[d] = v[e];
      }
    }
    __syncthreads();  // the next block writes tops, weights and sums again
  }
  if (kSplit || !row) return;
  const float share = keys_share(M, L, p.sinks, head);
#pragma unroll
  for (int o = 0; o < kOwn; ++o)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int d = 16 * (wave + o * kBlockWaves) + 4 * kg + e;
      if (d < p.v_dim) p.out[(static_cast<size_t>(t) * p.heads + head) * p.v_dim + d] = own[o][e] * share / L;
    }
}

// a workgroup per (head, token), a thread per element of the value
__global__ void __launch_bounds__(256) attention_f32_join_kernel(F32Attention p) {
  const int head = blockIdx.x, t = blockIdx.y, d = threadIdx.x;
  const int pos = p.positions[t], lo = first_key(pos, p.window, p.chunk);
  if (d >= p.v_dim) return;
  float M = -INFINITY, L = 0.f, sum = 0.f;
  for (int b = lo / kKeyBlock; b <= pos / kKeyBlock; ++b) {
    const float* block = p.partial + ((static_cast<size_t>(t) * p.heads + head) * p.blocks + b) * (p.v_dim + 2);
    float e0, e1;
    join_block(M, L, block[p.v_dim], block[p.v_dim + 1], e0, e1);
    sum = joined(sum, e0, block[d], e1);
  }
  const float share = keys_share(M, L, p.sinks, head);
  p.out[(static_cast<size_t>(t) * p.heads + head) * p.v_dim + d] = sum * share / L;
}

bool attention_f32_takes(int head_dim, int v_dim, int page_size, const void* k_pool, const void* v_pool) {
  return head_dim % 4 == 0 && page_size % 4 == 0 && reinterpret_cast<uintptr_t>(k_pool) % 16 == 0 &&
         reinterpret_cast<uintptr_t>(v_pool) % 16 == 0;
}

template <int D>
static void launch(const F32Attention& p, int n, int splits, int pairs, hipStream_t s) {
  const int per = p.heads / p.kv_heads;
  const dim3 grid(p.kv_heads * ((per + 15) / 16), n, splits);
  if (splits > 1) {
    attention_f32_kernel<D, true, false><<<grid, kWave * kBlockWaves, 0, s>>>(p, n);
    attention_f32_join_kernel<<<dim3(p.heads, n), (p.v_dim + kWave - 1) / kWave * kWave, 0, s>>>(p);
  } else {
    // Pairs where tokens by themselves would be workgroups for the chip one and a half times (heads of 64: two workgroups fit on a
    // compute unit) or three times (128: one does), else two tokens' chain of work is the longer one.  14 heads of 64 over 2,
    // at 165 / 200 / 509 / 2,000 tokens 11.3 / 14.1 / 37.7 / 366 us by themselves, 12.3 / 12.8 / 24.4 / 198 in pairs, 28 of 128 over 4 at
    // 130 / 200 / 509 / 2,000 31.6 / 38.8 / 114 / 1,237 and 35.1 / 36.6 / 98.8 / 955.  (Heads of more than 128 fill the registers.)
    // A token without a neighbour is the slower in that kernel, and so are heads of more than 96 over few keys (whole steps of
    // them: f32_pairs() in parts/attention.py), which only the caller knows of.
    constexpr bool kPairs = D <= 8;
    const bool wanted = pairs > 0 || (pairs < 0 && D <= 6);
    const auto kernel = wanted && per <= 8 && p.kv_heads * n > (D <= 6 ? 384 : 768) ? attention_f32_kernel<D, false, kPairs>
                                                                                    : attention_f32_kernel<D, false, false>;
    kernel<<<grid, kWave * kBlockWaves, 0, s>>>(p, n);
  }
}

void attention_f32(const F32Attention& p, int n, int splits, int pairs, hipStream_t s) {
  const int d = p.head_dim > p.v_dim ? p.head_dim : p.v_dim;
  // (heads of 40 in the kernel for 64, of 96 in that for 128: 500 tokens 34.7 us and 35.0 instead of 29.8 and 28.9)
  if (d <= 32)
    launch<2>(p, n, splits, pairs, s);
  else if (d <= 48)
    launch<3>(p, n, splits, pairs, s);
  else if (d <= 64)
    launch<4>(p, n, splits, pairs, s);
  else if (d <= 96)
    launch<6>(p, n, splits, pairs, s);
  else if (d <= 128)
    launch<8>(p, n, splits, pairs, s);
  else
    launch<16>(p, n, splits, pairs, s);
}

}  // namespace shk
