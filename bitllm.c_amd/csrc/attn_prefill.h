// attn_prefill.h -- causal attention of a prompt batch over the fp16 KV cache (attn_prefill.hip).
#pragma once

#include <hip/hip_fp16.h>

#include "hip_common.h"

namespace eif {

constexpr int kPfKeys = 32;          // keys of a staged tile
constexpr int kPfMinTiles = 4;       // fewest tiles of a share

struct PrefillAttn {
    const float *qkv;                // [n, ldqkv] rows q (rotated) | k | v
    int ldqkv;
    const __half *kc, *vc;           // the layer's cache [kv_head][seq_len][head_dim], positions 0 .. pos0 + n - 1 filled
    float *out;                      // [n, ldo], n_heads x head_dim
    int ldo;
    float *po, *pml;                 // shares of split blocks: rows of head_dim outputs, and of 2 (maximum, sum),
    size_t shares;                   // as many as these buffers hold
    int pos0, n, n_heads, n_kv, seq_len, head_dim;
};

// Rows of shares that a batch of n tokens may leave at any position of a cache of seq_len.
size_t prefill_attn_shares(int n, int n_heads, int n_kv, int seq_len);
int launch_attn_prefill(const PrefillAttn &a, hipStream_t st);

}  // namespace eif
