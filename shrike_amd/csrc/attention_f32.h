// The float32 attention on the matrix units (attention_f32.hip) as attention.hip launches it.
#pragma once

#include "common.h"

namespace shk {

constexpr int kKeyBlock = 256;  // keys whose maximum and sums are formed together

// partial: [tokens][heads][blocks][v_dim + 2] where the blocks of a token are formed apart (splits > 1)
struct F32Attention {
  const float *q, *k_pool, *v_pool, *sinks, *dist_bias;
  float *out, *partial;
  const int32_t *positions, *token_seq, *tables;
  int q_stride, heads, kv_heads, head_dim, v_dim, table_stride, page_size, num_pages, window, chunk, bias_rows, blocks;
  float scale, softcap;
};

bool attention_f32_takes(int head_dim, int v_dim, int page_size, const void* k_pool, const void* v_pool);
// pairs: shk_attention's
void attention_f32(const F32Attention& p, int n, int splits, int pairs, hipStream_t s);

}  // namespace shk
