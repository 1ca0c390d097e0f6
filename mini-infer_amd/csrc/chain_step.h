// chain_step.h -- the decoder step's stages several in one launch, for a
// caller that has every GEMM output of the step in hand before it starts
// (mi_decoder_chain_run).  Called by the host layer's DecoderChain, not part
// of the C ABI.
#pragma once

#include <stdint.h>

#include "mi_kernels.h"

namespace mi {

// hidden = table[ids] (* scale); normed = rmsnorm(hidden, w_in);
// hidden += attn;  post_normed = rmsnorm(hidden, w_post);
// hidden += mlp;   final_normed = rmsnorm(hidden, w_final),
// each step rounded to fp16 where the separate launches store it.  With
// w_attn / w_mlp (both or neither) attn and mlp are first normalised in place.
struct ChainRows {
    const int64_t* ids;
    const void* table;  // [vocab, D]
    void *hidden, *normed, *post_normed, *final_normed;  // [T, D]
    void *attn, *mlp;                                    // [T, D]
    const void *w_in, *w_post, *w_final, *w_attn, *w_mlp;  // [D]
    int64_t T, D, vocab;
    float scale, eps;
    int add_one;
};

// MI_OK, a hipError_t, or MI_ERR_UNSUPPORTED (nothing launched) for rows that
// are no whole number of aligned 16-byte vectors or longer than 8192: the
// caller then issues the stages one by one.  The buffers must not overlap
// one another (the caller checks).
int chain_rows(const ChainRows& r, void* stream);

// mi_rope_kv_scatter_f16 / mi_qk_norm_rope_kv_scatter_f16 (rope.hip), `wide` with
// up to 768 (head, slice) units per token.
int rope_kv_launch(void* q, void* k, const void* v, const void* q_bias, const void* k_bias,
                   const void* v_bias, const void* q_weight, const void* k_weight, float eps,
                   int add_one, const int64_t* positions, const float* inv_freq_host, int64_t T,
                   int64_t Hq, int64_t Hkv, int64_t head_dim, void* k_cache, void* v_cache,
                   int64_t layer, int64_t num_blocks, int64_t block_size,
                   const mi_kv_segment* segments, int num_segments, bool wide, void* stream);

// The whole step: the rows, the attention pre-processing into the cache, the
// activation and the sampling step, each with its entry point's arguments.
struct ChainStep {
    ChainRows rows;
    void *q, *k;
    const void *v, *q_bias, *k_bias, *v_bias, *q_weight, *k_weight;
    float qk_eps;
    const int64_t* positions;
    const float* inv_freq_host;
    int64_t Hq, Hkv, head_dim;
    void *k_cache, *v_cache;
    int64_t layer, num_blocks, block_size;
    const mi_kv_segment* segments;
    int num_segments;
    const void *gate, *up;
    void* act_out;
    int64_t act_n;
    int gelu;  // 0: SwiGLU, 1: GeGLU
    const void* logits;
    void* probs;
    int32_t* next_tokens;
    int64_t N, vocab;  // N = 0: the step without its sampling
    void* workspace;
    int64_t workspace_bytes;
};

// One launch for the step.  MI_OK, a hipError_t, or
// MI_ERR_UNSUPPORTED (nothing launched) for steps it does not take.  The buffers
// must not overlap one another but in the stages' own in-place forms (the caller
// checks).
int chain_step(const ChainStep& c, void* stream);

}  // namespace mi
