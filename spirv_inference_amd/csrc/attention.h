// Attention over any sequence length (head dim 64): attention_rows, attention_fused and the
// decoder's prompt pass.
#pragma once

#include "common.h"

namespace shp {

// out[b, i, h, :] = softmax_t(q[b, i, h, :] . k[b, t, h / group, :] * scale (+ mask[t])) . v
// Element strides: *_b per batch, *_h per head (q, out: query head; k, v: KV head), *_r per row.
// Rows are 64 contiguous floats, 16-byte aligned.
struct AttnArgs {
    const float *q, *k, *v;
    const float* mask;  // [n_keys] additive, or null (not with causal)
    float* out;
    int64_t q_b, q_h, q_r, k_b, k_h, k_r, v_b, v_h, v_r, o_b, o_h, o_r;
    int batch, kv_heads, group;  // group query heads share one KV head
    int n_queries, n_keys;
    int causal;  // 1: query i sees keys t <= pos0 + i
    int pos0;
    float scale;
};

int attention_launch(hipStream_t s, const AttnArgs& a);

}  // namespace shp
