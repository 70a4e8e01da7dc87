// Device steps of a block of prompt tokens (prefill) that are not linear layers: embedding,
// head norms with RoPE and the cache rows, and causal attention.  Launchers of attn_rows.hip;
// every kernel keeps the host step's operation order (see there).
#ifndef BNNE_ATTN_ROWS_H
#define BNNE_ATTN_ROWS_H

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bnne {

constexpr uint32_t kRowsHeadDim = 128;  // head_dim of these kernels

struct AttnRows {
    uint32_t rows, pos0;            // the block's tokens are at positions pos0 .. pos0 + rows - 1
    uint32_t heads, kv_heads, kv_dim;
    float eps, scale;
    float *q, *k, *v;               // [rows][heads * 128], [rows][kv_dim]: the projections (q is overwritten)
    const float *q_gain, *k_gain;   // [128]
    const float *cosv, *sinv;       // [positions][64], position 0
    float *kc, *vc;                 // the layer's cache rows, position 0
    float* scores;                  // [heads][rows][score_pitch]
    uint32_t score_pitch;           // a multiple of 64, at least pos0 + rows
    float* y;                       // [rows][heads * 128]
    int* err;                       // set to 1 by a failed check
};

// x[r] = the embedding row of tokens[r]; clears the error word and the logits flag (where not null).
void launch_embed_rows(hipStream_t stream, const int32_t* tokens, uint32_t rows, const uint8_t* bits,
                       const uint16_t* scales, uint32_t C, float* x, int* err, int* logit_bad);
// Head norms, RoPE, cache rows, scores, softmax and the weighted values of one layer.
void launch_attn_rows(hipStream_t stream, const AttnRows& a);

}  // namespace bnne

#endif
