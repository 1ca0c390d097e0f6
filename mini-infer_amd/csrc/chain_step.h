// chain_step.h -- the decoder step's row-wise stages as one launch, for a
// caller that has every GEMM output of the step in hand before it starts
// (mi_decoder_chain_run).  Called by the host layer's DecoderChain, not part
// of the C ABI.
#pragma once

#include <stdint.h>

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

}  // namespace mi
