// What the runtime's reference sequence (model.cpp) launches beside the C ABI:
// the Q5_0 / Q8_0 GEMVs of a decode step with the work around them in the same
// launch (gemv_q8_0_q5_0.hip), RoPE with the cache append, and the argmax over
// many workgroups (decode_ops.hip).
#pragma once
#include <stdint.h>

#include "taraference_hip.h"

// Rows that the fused forms take: an even number of blocks, at most 64.
bool tf_b32_norm_fits(int n_rows);

// q, k (Q5_0) and v (Q8_0, dword-aligned columns) of rmsnorm(x) * norm_w, each
// with its bias (bq and bk both or neither).  x, norm_w 16-byte aligned.
int tf_b32_norm_qkv(const float* x, const float* norm_w, float eps, const uint8_t* wq,
                    const uint8_t* wk, const uint8_t* wv, float* q, float* k, float* v,
                    const float* bq, const float* bk, const float* bv, int n_rows, int n_q, int n_k,
                    int n_v, int cb_qk, int cb_v, tf_stream_t stream);
// h = silu(gate n) * (up n) for n = rmsnorm(x) * norm_w, both Q5_0.
int tf_b32_norm_gate_up(const float* x, const float* norm_w, float eps, const uint8_t* gate,
                        const uint8_t* up, float* h, int n_rows, int n_cols, int col_bytes,
                        tf_stream_t stream);
// x += wo a (Q5_0) for the attention output a given as split-KV partials
// (tf_flash_decode_partial's layout).
bool tf_b32_flash_out_fits(int n_head, int head_dim, int parts);
int tf_b32_flash_out(const uint8_t* w, const float* partial, int n_head, int head_dim, int parts,
                     float* x, int n_cols, int col_bytes, tf_stream_t stream);
// q and k heads rotated (NeoX, in place), k and v appended to the f16 caches at
// row pos (pos_dev[0] if given).
int tf_rope_append(float* q, float* k, const float* v, uint16_t* k_cache, uint16_t* v_cache,
                   int n_head, int n_kv, int head_dim, int pos, const int* pos_dev, float theta,
                   tf_stream_t stream);
// The argmax of n logits as keys in slots (TF_ARGMAX_SLOTS, all of them clear), to
// be taken by tf_argmax_key_finalize or the step that advances.
int tf_argmax_keys(const float* x, int n, unsigned long long* slots, tf_stream_t stream);
