// A decoding step of one sequence as one launch (token.hip); the host side is in inference.hip.
#pragma once
#include "backend.h"
#include <algorithm>
#include <stddef.h>

namespace lmhip {

constexpr int TOKEN_MAX_LAYERS = 48;
constexpr int TOKEN_KEYS = 256;          // keys of a context that the attention inside takes

struct TokenShape { int D, IS, Hq, Hkv, hd, NL, V; };

// device addresses of a layer: weights (rows of F16, or codes with their scales behind *_d), norm weights (0 where there is
// none; g_post_attn, g_post_ff: norms of the branches), caches [Hkv, max_seq, hd], (cos, sin) of all positions
struct TokenLayer {
    uint64_t qkv, qkv_d, o, o_d, gu, gu_d, down, down_d;
    uint64_t g_in, g_post_attn, g_ff, g_post_ff, g_q, g_k, kc, vc, rope;
};

struct TokenArgs {
    const uint64_t *layers;              // NL x TokenLayer
    const float *emb_row, *g_final;
    const void *head, *head_d;
    unsigned long long *qkv_w, *att_w, *o_w, *h_w, *down_w, *best_w;          // words (token_words)
    float *logits, *logits_host;         // logits_host: pinned copy, or null
    int *best_host, *fail;               // pinned; best_host null: no argmax
    uint64_t ticks;                      // of the 100 MHz clock that a step may wait
    uint32_t tag;                        // NL + 1 tags from here on, none of which the words hold
    int NL, D, IS, Hq, Hkv, hd, max_seq, V, pos, gemma;
    float emb_scale, eps, scale;
};

bool token_fits(const TokenShape &s);
bool token_pays(const TokenShape &s, int q8);            // among those that fit
// 64-bit words that a state needs for its hand-overs, zero before the first step; with a and base: their places
size_t token_words(const TokenShape &s, TokenArgs *a, unsigned long long *base);
void launch_token(const TokenArgs &a, const TokenShape &s, int q8);

// infer_kernels.hip: addresses of a Q8_0 matrix's codes and scales in an image that stays with the buffer (false: it has none that stays)
bool q8_rows_of(MetalBuf *W, int rows, int cols, const void **codes, const void **scales);

}  // namespace lmhip
