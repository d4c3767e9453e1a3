// Internal prefill entry points used by the decode runtime (model.cpp): the
// GEMMs on x images with the glue fused around them (prefill_gemm.hip), the
// embedding rows and the attention (prefill.hip).
#pragma once
#include <stdint.h>

#include "taraference_hip.h"

// A prompt's GEMMs read x as images: its two f16 parts in the order in which
// the matrix cores take them, made once by the kernel that produces x (or by
// tf_pg_image from f32 rows).  Bytes for n_tok rows of n_rows values:
size_t tf_pg_image_bytes(int n_rows, int n_tok);
int tf_pg_image(const float* x, uint8_t* img, int n_rows, int n_tok, tf_stream_t stream);

// A GEMM's output as n_split slices of K, to be added in order: slice z of
// value i at p[z * stride + i].
struct TfPgPart {
    const float* p;
    int n_split;
    long long stride;
};

// x[t] += part[t] (part may be null), then img = rmsnorm(x) * w.
// n % 256 == 0; w at any multiple of 4 bytes.
int tf_pg_norm_image(float* x, const TfPgPart* part, const float* w, float eps, uint8_t* img, int n,
                     int n_tok, tf_stream_t stream);
// x[row] += part[row], rows of n.
int tf_pg_add_row(float* x, const TfPgPart& part, int row, int n, tf_stream_t stream);
// part = W x for Q4_K (block_bytes 144), raw (210) or compact (212) Q6_K
// weights; the slices in ws (at least n_tok * n_cols floats).
int tf_pg_gemm(const uint8_t* w, int block_bytes, const uint8_t* img, int n_rows, int n_cols,
               int col_bytes, int n_tok, float* ws, size_t ws_floats, TfPgPart* part,
               tf_stream_t stream);
// The same for q, k and v side by side in rows of n_cols[0] + [1] + [2].
int tf_pg_qkv(const uint8_t* const w[3], const int block_bytes[3], const int n_cols[3],
              const int col_bytes[3], const uint8_t* img, int n_rows, int n_tok, float* ws,
              size_t ws_floats, TfPgPart* part, tf_stream_t stream);
// biases, NeoX RoPE of q and k at positions pos0 + t, q rows to q_out, k and v
// appended to the f16 caches at rows pos0 + t.
int tf_pg_qkv_post(const TfPgPart& part, const float* bq, const float* bk, const float* bv,
                   float* q_out, uint16_t* k_cache, uint16_t* v_cache, int n_head, int n_kv,
                   int head_dim, int pos0, int n_tok, float theta, tf_stream_t stream);
// out = silu(gate x) * (up x), both Q4_K.
int tf_pg_gate_up(const uint8_t* gate, const uint8_t* up, const uint8_t* img, float* out,
                  int n_rows, int n_cols, int col_bytes, int n_tok, tf_stream_t stream);
int tf_attn_prefill_any(const float* q, const uint16_t* k_cache, const uint16_t* v_cache,
                        float* out, int n_head, int n_kv, int head_dim, int pos0,
                        const int* pos0_dev, int n_q, float scale, tf_stream_t stream);
// out[t] = embedding row of tokens_dev[t] (Q4_K 144 or Q6_K 210 blocks).
int tf_pf_embed(const uint8_t* table, int block_bytes, const int* tokens_dev, float* out,
                int n_rows, int col_bytes, int n_tok, tf_stream_t stream);
// g = silu(g) * u over n values.
int tf_pf_silu_mul(float* g, const float* u, long long n, tf_stream_t stream);
