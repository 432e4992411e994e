// bfloat16 attention of prompt portions over the paged cache, 32 rows a wavefront.
//
// A row is one query of one head.  The heads that share a key/value head read the same keys, so a workgroup of eight
// wavefronts takes all of them for a run of queries: 256 rows, whatever the heads of a group (36 queries of 7 heads, 51
// of 5).  The products are formed transposed with v_mfma_f32_32x32x16_bf16 (S^T = K Q^T, O^T += V^T P^T): a lane owns
// half of a row's scores, and P goes from one product into the next without leaving its lane.
//
// Chunks of 64 keys.  Keys and values go from the pages straight into LDS, two chunks ahead; a tile of 32 keys has its
// scores formed while the softmax arithmetic of the tile before runs on the vector units, and is multiplied with its values
// under the tile after.
//   keys    [group of 16][32 elements] units of 1 KiB as in the page (64 bytes a key): piece c of a key at place c ^ (key / 4),
//   values  [group of 16][32 elements] units of 32 bytes an element: piece c at place c ^ (element / 8 % 2),
// so that the 16 lanes that LDS serves at once meet no bank conflicts.  Row i = 8 g + 4 h + r of a score tile is key
// 16 (g / 2) + 8 h + 4 (g % 2) + r of its 32: the lane's scores are then, in order, the eight keys that it has to bring
// to the second product.
//
// What bounds it: the vector units' issue, about 170 instructions a wavefront and tile, 64 of them the rescaling of o in
// every tile (a branch around it costs as much in copies), beside 16 multiplications: the matrix units are busy 40 % of
// the time.  Weights relative to a reference that rarely moves would need no rescaling (118 us where this kernel took 137, 512
// queries at 12,001), but are a tenth less exact: the largest would no longer be 1.
// Against the kernel with 16 queries a wavefront, which reads every operand from LDS twice as often, 28 heads over 4: 512
// queries at 12,001 148 us -> 123 alone and 156 -> 144 a layer in a model's pass; alone, at 31,000 335 -> 279, at 3,584 61 -> 55, at
// 1,536 40 -> 40, at 0 21 -> 25 (fewer, longer workgroups); 4,096 from 0 183 -> 151, 2,048 69 -> 74.  Where portions fill few
// of a workgroup's rows it loses (64 of 8 queries at 2,000: 60 -> 80).  The bits are the same with the same shares.
#include "attention_rows.h"
#include "gemm_wide.h"
#include "mfma_tile.h"

namespace shk {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float halves_max(float v) {
  const unsigned b = __builtin_bit_cast(unsigned, v);
  const auto halves = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  return fmaxf(bits_as_float(halves[0]), bits_as_float(halves[1]));
}
__device__ __forceinline__ float halves_sum(float v) {
  const unsigned b = __builtin_bit_cast(unsigned, v);
  const auto halves = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  return bits_as_float(halves[0]) + bits_as_float(halves[1]);
}

template <int D>
__global__ void __launch_bounds__(8 * kWave) __attribute__((amdgpu_waves_per_eu(2, 2)))
    attention_rows_kernel(const bf16* __restrict__ q, int q_stride, bf16* __restrict__ out, int heads, int kv_heads, int queries,
                          const int32_t* __restrict__ cu_q, const int32_t* __restrict__ ctx_lens, const int32_t* __restrict__ wg_seq,
                          const int32_t* __restrict__ wg_q0, const int32_t* __restrict__ tables, int table_stride,
                          const bf16* __restrict__ k_pool, const bf16* __restrict__ v_pool, int page_size, uint32_t page_magic,
                          int window, int block, float scale, float* __restrict__ partial, int nsplit, int first_token,
                          int partial_rows, const float* __restrict__ sinks) {
  constexpr int KS = D / 16, DB = D / 32;           // steps of a score tile; blocks of 32 elements
  constexpr int kSide = 4 * DB, kLoads = kSide / 8;  // units of a chunk's keys (and of its values); a wavefront's of each
  constexpr int kRing = 4, kBytes = kSide * 1024;  // chunks; bytes of a chunk's keys
  static_assert(kLoads >= 1 && kSide % 8 == 0, "a wavefront loads whole units");
  __shared__ u32x4 mem[(2 * kRing * kBytes + 2 * DB * 1024) / 16];  // keys, values, a tile's values of zero
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int col = lane % 32, half = lane / 32;
  const PageDiv pd{page_size, page_magic};
  // workgroups start in the order of the host's list (every key/value head of an entry side by side)
  const int z = blockIdx.x % nsplit;  // which share of the entry's keys
  const int wg = blockIdx.x / (nsplit * kv_heads), kvh = (blockIdx.x / nsplit) % kv_heads;
  const int seq = wg_seq[wg], q0 = wg_q0[wg];
  const int group = heads / kv_heads;
  const int tok0 = cu_q[seq], q_len = cu_q[seq + 1] - tok0;
  const int start = ctx_lens[seq] - q_len;  // position of the portion's first token
  const int q_end = q0 + queries < q_len ? q0 + queries : q_len;
  const int32_t* table = tables + static_cast<size_t>(seq) * table_stride;

  // what the workgroup reads: keys lo_min .. pos_max, in chunks of 64 from key_begin on
  const int pos_min = start + q0, pos_max = start + q_end - 1;
  const int lo_min = first_key(pos_min, window, block), lo_max = first_key(pos_max, window, block);
  const int key_begin = lo_min & ~63;
  const int nchunks = (pos_max - key_begin) / 64 + 1;
  const int per_split = (nchunks + nsplit - 1) / nsplit;
  const int c_first = z * per_split;
  const int c_end = c_first + per_split < nchunks ? c_first + per_split : nchunks;

  // the lane's row (both halves of the wavefront hold the same 32); a lane without one reads no key
  const int row = wave * 32 + col, qi = q0 + row / group, head = kvh * group + row % group;
  const bool mine = qi < q_end;
  const int q_pos = mine ? start + qi : -1, q_lo = first_key(q_pos, window, block);
  u32x4 qf[KS];
  {
    const bf16* src = q + static_cast<size_t>(tok0 + (mine ? qi : q0)) * q_stride + static_cast<size_t>(mine ? head : kvh * group) * D + half * 8;
#pragma unroll
    for (int st = 0; st < KS; ++st) qf[st] = *reinterpret_cast<const u32x4*>(src + st * 16);
  }
  float m = -INFINITY, l = 0.f;  // base-2 logarithm of the maximum; the lane's share of the sum
  f32x16 o[DB];                  // element db * 32 + 8 g + 4 half + r of the row in register g * 4 + r
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[db][r] = 0.f;
  const float scale2 = scale * 1.4426950408889634f;

  // ---- what a wavefront loads of a chunk: units wave * kLoads .. of the keys and of the values, all of one group of 16
  const unsigned base = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)&mem[0]));
  const int my_group = wave * kLoads / DB, my_block = wave * kLoads % DB;
  unsigned koff[kLoads], voff[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int key = lane / 4, e = lane / 2;
    koff[i] = static_cast<unsigned>((my_block + i) * page_size * 64 + key * 64 + ((lane % 4) ^ (key / 4)) * 16);
    voff[i] = static_cast<unsigned>(((my_block + i) * 32 + e) * page_size * 2 + ((lane % 2) ^ ((e / 8) % 2)) * 16);
  }
  // the group of 16 keys that stands for this wavefront's of a chunk: one that the sequence holds and the workgroup reads
  auto group_key = [&](int chunk) __attribute__((always_inline)) {
    int key = key_begin + 64 * (chunk < nchunks ? chunk : nchunks - 1) + 16 * my_group;
    key = key > lo_min ? key : lo_min;
    key = key < pos_max ? key : pos_max;
    return key & ~15;
  };
  // a chunk's group: its page, asked for a step before the others, where the head's part of that page begins, its slot
  struct Group {
    uint64_t at;
    int slot;
  };
  auto page_of = [&](int chunk) __attribute__((always_inline)) { return table[__builtin_amdgcn_readfirstlane(pd.div(group_key(chunk)))]; };
  const unsigned head_bytes = static_cast<unsigned>(page_size) * (2 * D);
  auto group_of = [&](int chunk, int page) __attribute__((always_inline)) {
    const unsigned part = __builtin_amdgcn_readfirstlane(page) * static_cast<unsigned>(kv_heads) + kvh;
    return Group{static_cast<uint64_t>(part) * head_bytes, __builtin_amdgcn_readfirstlane(pd.mod(group_key(chunk)))};
  };
  auto load_k = [&](int slot, Group g) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i)
      SHK_LOAD_TO_LDS(base + slot * kBytes + (wave * kLoads + i) * 1024, koff[i], reinterpret_cast<const char*>(k_pool) + g.at + g.slot * 64);
  };
  auto load_v = [&](int slot, Group g) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i)
      SHK_LOAD_TO_LDS(base + (kRing + slot) * kBytes + (wave * kLoads + i) * 1024, voff[i], reinterpret_cast<const char*>(v_pool) + g.at + g.slot * 2);
  };

  // ---- where this lane's operands lie
  const char* lds = reinterpret_cast<const char*>(&mem[0]);
  const int key = 16 * (col / 16) + 8 * (col / 4 % 2) + 4 * (col / 8 % 2) + col % 4;  // of a tile's 32: its row `col`
  const int turn = key / 4 % 4;
  const int kat = (key / 16) * DB * 1024 + (key % 16) * 64;
  const int kpiece[2] = {(half ^ turn) * 16, ((2 + half) ^ turn) * 16};
  const int vat = kRing * kBytes + col * 32 + (half ^ ((col / 8) % 2)) * 16;
  auto key_operand = [&](int from, int st) __attribute__((always_inline)) {  // from: where the tile's keys begin
    return *reinterpret_cast<const u32x4*>(lds + from + kat + st / 2 * 1024 + kpiece[st % 2]);
  };
  auto value_operand = [&](int from, int i) __attribute__((always_inline)) {  // i: (keys of 16) * DB + block of elements
    return *reinterpret_cast<const u32x4*>(lds + from + vat + i * 1024);
  };
  auto score = [&](f32x16& s, u32x4 kf, int st) __attribute__((always_inline)) {
    s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kf), __builtin_bit_cast(bf16x8, qf[st]), s, 0, 0, 0);
  };
  auto add_values = [&](u32x4 vf, const bf16x8 (&p)[2], int i) __attribute__((always_inline)) {
    o[i % DB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, vf), __builtin_bit_cast(bf16x8, p[i / DB]), o[i % DB], 0, 0, 0);
  };
  // Values of keys outside [lo_min, pos_max] get weights of 0, but their slots in the page may hold anything: a wavefront
  // clears what it has loaded of them for chunk c.
  auto clear_values = [&](int c, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      u32x4* at = &mem[((kRing + slot) * kBytes + (wave * kLoads + i) * 1024) / 16 + lane];
      const int first = key_begin + 64 * c + 16 * my_group + 8 * ((lane % 2) ^ ((lane / 16) % 2));
      u32x4 v = *at;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool a = first + 2 * e >= lo_min && first + 2 * e <= pos_max;
        const bool b = first + 2 * e + 1 >= lo_min && first + 2 * e + 1 <= pos_max;
        v[e] &= (a ? 0x0000ffffu : 0u) | (b ? 0xffff0000u : 0u);
      }
      *at = v;
    }
  };

  // Of the tile before, whose values begin at `before`.  The first tile's product with it is 0 times 0: with values that are
  // there, infinities among them, 0 times those would be NaN.
  bf16x8 weights[2];
  int before = kRing * kBytes;
  for (int i = threadIdx.x; i < 2 * DB * kWave; i += 8 * kWave) mem[2 * kRing * kBytes / 16 + i] = u32x4{0, 0, 0, 0};
#pragma unroll
  for (int e = 0; e < 8; ++e) weights[0][e] = weights[1][e] = static_cast<__bf16>(0.f);

  if (c_first < c_end) {  // the same for every wavefront of the workgroup
    // Loads in the order in which they are waited for: K(c), V(c), K(c + 1), V(c + 1), ...  Step c reads V(c - 1), V(c),
    // K(c) and K(c + 1), so behind its barrier K(c - 1) and V(c - 2) are read no more: K(c + 3) and V(c + 2) go into
    // their places.  What it reads was asked for two steps before.
    Group g2, g3;  // of chunks c + 2 and c + 3
    int page = page_of(c_first + 4);
    {
      const int p0 = page_of(c_first), p1 = page_of(c_first + 1), p2 = page_of(c_first + 2), p3 = page_of(c_first + 3);
      const Group g0 = group_of(c_first, p0), g1 = group_of(c_first + 1, p1);
      g2 = group_of(c_first + 2, p2), g3 = group_of(c_first + 3, p3);
      load_k(0, g0);
      load_v(0, g0);
      load_k(1, g1);
      load_v(1, g1);
      load_k(2, g2);
    }
    const int last_plain = (pos_min + 1 - key_begin) / 32 - 1, tiles = (pos_max - key_begin) / 32 + 1;
    const int first_plain = lo_max > key_begin ? (lo_max - key_begin + 31) / 32 : 0;
    const int t_end = 2 * c_end < tiles ? 2 * c_end : tiles;
    constexpr int M = KS + 2 * DB, kAhead = 6;  // multiplications of a tile; operands asked for ahead
    f32x16 s;      // scores of the tile to come, as they leave the matrix unit
    float sc[16];  // the same as base-2 logarithms
    float mx = 0.f, alpha = 1.f;  // their maximum; what o has to be multiplied by for the reference of the tile before
    auto take = [&](int e) __attribute__((always_inline)) {
      sc[e] = s[e] * scale2;
      if (e == 1) mx = fmaxf(sc[0], sc[1]);
      if (e > 1 && e % 2) mx = max3(mx, sc[e - 1], sc[e]);
    };
    SHK_MEET_WITH_LOADS(4 * kLoads);
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
    for (int st = 0; st < KS; ++st) score(s, key_operand(0, st), st);
#pragma unroll
    for (int e = 0; e < 16; ++e) take(e);
    // One tile of 32 keys, whose scores are in sc, in every turn: its softmax arithmetic, and between its instructions the
    // scores of the next tile and the tile before's product with its values.  Nothing moves across sched_barrier.
    // o is multiplied by alpha in every turn: a branch around that makes the compiler copy all of o instead.
    for (int t = 2 * c_first; t < t_end; ++t) {
      const int c = t / 2, odd = t % 2, kb = key_begin + 32 * t;
      const unsigned at = (c - c_first) % kRing;  // the chunk's place in the rings
      if (!odd) {
        SHK_MEET_WITH_LOADS(2 * kLoads);
        if (kb < lo_min || kb + 63 > pos_max) {
          clear_values(c, at);
          __syncthreads();
        }
        load_k((at + 3) % kRing, g3);
        load_v((at + 2) % kRing, g2);
        g2 = g3;
      }
      // (the scores behind the last tile are of keys that are there, and never used)
      const unsigned next = odd ? (at + 1) % kRing * kBytes : at * kBytes + 2 * DB * 1024;
      u32x4 operand[M];
      auto ask = [&](int q) __attribute__((always_inline)) {
        operand[q] = q < KS ? key_operand(next, q) : value_operand(before, q - KS);
      };
#pragma unroll
      for (int q = 0; q < kAhead; ++q) ask(q);
      if (t > last_plain || t < first_plain) {  // some query does not read all of it
        // register g * 4 + r is key 16 (g / 2) + 8 half + 4 (g % 2) + r
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int key_at = kb + e / 8 * 16 + 8 * half + e % 8;
          if (key_at > q_pos || key_at < q_lo) sc[e] = -INFINITY;
        }
        mx = fmaxf(sc[0], sc[1]);
#pragma unroll
        for (int e = 2; e < 16; e += 2) mx = max3(mx, sc[e], sc[e + 1]);
      }
      const float m_new = fmaxf(m, halves_max(mx));
      const float m_safe = m_new == -INFINITY ? 0.f : m_new;  // (a row that has read no key yet)
      const float alpha_new = __builtin_amdgcn_exp2f(m - m_safe);
      m = m_new;
      float sum[2] = {0.f, 0.f};
      bf16x8 p[2];
      auto weigh = [&](int i) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 2 * i; e < 2 * i + 2; ++e) {
          const float w = __builtin_amdgcn_exp2f(sc[e] - m_safe);
          sum[e % 2] += w;
          p[e / 8][e % 8] = static_cast<__bf16>(w);
        }
        // (here, not where the compiler would sink it to: behind the multiplications)
        asm volatile("" : "+v"(sum[0]), "+v"(sum[1]), "+v"(p[i / 4]));
      };
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
      for (int q = 0; q < M; ++q) {
        if (q + kAhead < M) ask(q + kAhead);
        if (q < KS) {
          score(s, operand[q], q);
#pragma unroll
          for (int r = q * 16 * DB / KS; r < (q + 1) * 16 * DB / KS; ++r) o[r / 16][r % 16] *= alpha;
        } else {
          add_values(operand[q], weights, q - KS);
        }
        // the weights in the middle of the turn, the next tile's scores when they have left the matrix unit
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (M / 8 + i * M / 16 == q) weigh(i);
#pragma unroll
        for (int e = 0; e < 16; ++e)
          if (M * 5 / 8 + e * (M * 3 / 8) / 16 == q) take(e);
        __builtin_amdgcn_sched_barrier(0);
      }
      l = l * alpha_new + (sum[0] + sum[1]);
      alpha = alpha_new;
      weights[0] = p[0], weights[1] = p[1];
      before = at * kBytes + odd * 2 * DB * 1024;
      if (odd) {  // where the loads of the next step come from
        g3 = group_of(c + 4, page);
        page = page_of(c + 5);
      }
    }
#pragma unroll
    for (int db = 0; db < DB; ++db) o[db] *= alpha;
#pragma unroll
    for (int i = 0; i < 2 * DB; ++i) add_values(value_operand(before, i), weights, i);
    SHK_WAIT_LOADS(0);  // no load may arrive in LDS that the workgroup has given back
  }

  float total = halves_sum(l);
  if (!mine) return;
  if (nsplit > 1) {
    // a share's result, for attention_merge_kernel: O [row][share][D], then (maximum, sum) [row][share][2]
    const size_t at = static_cast<size_t>(tok0 + qi - first_token) * heads + head;
    float* dst = partial + (at * nsplit + z) * D + 4 * half;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4*>(dst + db * 32 + g * 8) = f32x4{o[db][g * 4], o[db][g * 4 + 1], o[db][g * 4 + 2], o[db][g * 4 + 3]};
    if (!half)
      *reinterpret_cast<float2*>(partial + static_cast<size_t>(partial_rows) * nsplit * D + (at * nsplit + z) * 2) = make_float2(m, total);
    return;
  }
  if (sinks) total += __builtin_amdgcn_exp2f(sinks[head] * 1.4426950408889634f - m);
  const float inv = 1.f / total;
  bf16* dst = out + (static_cast<size_t>(tok0 + qi) * heads + head) * D + 4 * half;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      bf16x4 v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = static_cast<__bf16>(o[db][g * 4 + r] * inv);
      *reinterpret_cast<bf16x4*>(dst + db * 32 + g * 8) = v;
    }
}

bool launch_attention_rows(int head_dim, int workgroups, hipStream_t s, const bf16* q, int q_stride, bf16* out, int heads, int kv_heads,
                           int queries, const int32_t* cu_q, const int32_t* ctx_lens, const int32_t* wg_seq, const int32_t* wg_q0,
                           const int32_t* tables, int table_stride, const bf16* k_pool, const bf16* v_pool, int page_size, int window,
                           int block, float scale, float* partial, int nsplit, int first_token, int partial_rows,
                           const float* sinks) {
  const uint32_t magic = static_cast<uint32_t>(((1ull << 32) + page_size - 1) / page_size);
  if (head_dim != 64 && head_dim != 128) return false;
  const auto kernel = head_dim == 64 ? attention_rows_kernel<64> : attention_rows_kernel<128>;
  kernel<<<workgroups, 8 * kWave, 0, s>>>(q, q_stride, out, heads, kv_heads, queries, cu_q, ctx_lens, wg_seq, wg_q0, tables, table_stride,
                                          k_pool, v_pool, page_size, magic, window, block, scale, partial, nsplit, first_token,
                                          partial_rows, sinks);
  return true;
}

}  // namespace shk
