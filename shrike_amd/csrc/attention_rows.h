// Prompt attention with 32 rows a wavefront (attention_rows.hip).
#pragma once

#include "common.h"

namespace shk {

// Rows (a query of one head each) that a workgroup serves.
constexpr int kAttentionRows = 256;

// The arguments of attention_prefill_shared's kernels; workgroups serve `queries` consecutive queries of every head of
// a key/value head.  False: the head size is not served.
bool launch_attention_rows(int head_dim, int workgroups, hipStream_t s, const bf16* q, int q_stride, bf16* out, int heads, int kv_heads,
                           int queries, const int32_t* cu_q, const int32_t* ctx_lens, const int32_t* wg_seq, const int32_t* wg_q0,
                           const int32_t* tables, int table_stride, const bf16* k_pool, const bf16* v_pool, int page_size, int window,
                           int block, float scale, float* partial, int nsplit, int first_token, int partial_rows,
                           const float* sinks);

}  // namespace shk
