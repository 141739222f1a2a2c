// The decoder's prompt pass: all prompt positions of a chunk at once, so a chunk reads the
// weights once where the token-by-token feed reads them once per position.
#pragma once

#include "common.h"

namespace shp {

constexpr int kPrefillRows = 512;   // prompt positions per chunk (the ids ride in the arguments)
constexpr int kSkinnyRows = 64;     // rows up to which the weight-streaming product is used
constexpr int kSkinnySplits = 8;    // K ranges of a skinny product at most

struct PrefillIds {
    int32_t id[kPrefillRows];
};

// What a skinny product does with its sums.
enum SkinnyOut {
    SK_PARTIAL = 0,  // out[s][m][n]: the s-th K range's sums, added by the reader
    SK_SWIGLU = 1,   // out[m][n / 2] = silu(even n) * odd n (one K range)
};

// K ranges the product of M <= 64 rows with N weight rows of K is cut into.
int skinny_splits(int N, int K);
// x [M][K] times w [N][K]^T, M <= 64, K % 4 == 0, N % 8 == 0, 16-byte aligned.
int skinny_launch(hipStream_t s, const float* x, int M, const float* w, int N, int K, int mode,
                  int splits, float* out);

int prefill_embed_launch(hipStream_t s, const float* embed, int hidden, const PrefillIds& ids,
                         int rows, float* x);
// x += sum of `splits` partials (none if 0), stored to xout; h = rmsnorm(x) * w.
int prefill_norm_launch(hipStream_t s, const float* x, const float* part, int splits, float* xout,
                        const float* w, float eps, float* h, int rows, int hidden);
// Sums the qkv partials, rotates q and k at position pos0 + row, writes q [rows][heads * 64] and
// appends k and v to the layer's caches [kv][max_seq][64].
int prefill_rope_launch(hipStream_t s, const float* part, int splits, float* q, float* k_cache,
                        float* v_cache, int rows, int n_heads, int n_kv, int max_seq, int pos0,
                        float theta);
// act[m][n] = silu(gu[m][2n]) * gu[m][2n + 1].
int prefill_swiglu_launch(hipStream_t s, const float* gu, float* act, int rows, int ffn);
// Greedy argmax of each row (lowest index on ties) into log[0 .. rows); the last row's logits go
// to last_logits (when not null), its argmax to *token and pos to *pos / *step.
int prefill_argmax_launch(hipStream_t s, const float* logits, int rows, int vocab, int32_t* log,
                          float* last_logits, int32_t* token, int32_t* pos, int32_t* step,
                          int new_pos);

}  // namespace shp
