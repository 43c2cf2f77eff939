/*
 * miniep_amd_model.h -- the part of the C ABI that the transformer around the
 * MoE block calls (the MoE block itself: miniep_amd.h, whose conventions on
 * pointers, streams, return codes and dtypes hold here too).
 */
#ifndef MINIEP_AMD_MODEL_H
#define MINIEP_AMD_MODEL_H

#include "miniep_amd.h"

#ifdef __cplusplus
extern "C" {
#endif

/* ------------------------------------------------------------------------
 * The transformer around the MoE block (modeling.py:55-80,146-197).
 *
 * mep_add_norm: h_out = h + round(delta * mult) with each step rounded to
 * `dtype` (delta NULL: h_out is not written and stands for h), x_out =
 * weight * (h_out / sqrt(mean(h_out^2) + eps)) in fp32, rounded to `dtype`.
 * h_out may be h.  (n_rows, hidden) rows, hidden a multiple of 16 bytes, at
 * most 4096.
 *
 * mep_attention: rotate-half RoPE of q and k at positions start .. start+t-1
 * of the tables cos / sin (n_positions, head_dim) fp32; rotated keys and the
 * values go into the caches (batch, n_kv_heads, max_len, head_dim) fp32 at
 * those positions, and query i of each sequence attends positions 0 ..
 * start+i (scores times `scale`), all in fp32.  q (batch*t, n_heads*head_dim),
 * k / v (batch*t, n_kv_heads*head_dim), out like q, in `dtype`.
 * Supported: head_dim 64, n_heads / n_kv_heads in {1, 2, 4}.  One launch for
 * t = 1, two otherwise.
 * ---------------------------------------------------------------------- */
int mep_add_norm(const void* h, const void* delta, float mult, const void* weight, float eps,
                 int64_t n_rows, int32_t hidden, int32_t dtype, void* h_out, void* x_out, void* stream);

int mep_attention(const void* q, const void* k, const void* v, const float* cos, const float* sin,
                  int64_t n_positions, int32_t batch, int32_t t, int32_t n_heads, int32_t n_kv_heads,
                  int32_t head_dim, int64_t start, int64_t max_len, float scale, int32_t dtype,
                  float* k_cache, float* v_cache, void* out, void* stream);

/* ------------------------------------------------------------------------
 * The attention half of Block.forward (modeling.py:186-192) for at most 32
 * rows (batch * t) of a bf16 model, as one call (4 launches for t = 1):
 *   h1 = h + round(delta * mult)      (delta NULL: h1 = h)
 *   q, k, v = rms_norm(h1; norm1) @ {wq, wk, wv}^T
 *   o = attention of them (mep_attention: RoPE, cache write, causal)
 *   h_out = h1 + round(round(o @ wo^T) * mult),  x_out = rms_norm(h_out; norm2)
 * Each projection is rounded to bf16, sums are fp32.  wq (n_heads*head_dim,
 * hidden), wk / wv (n_kv_heads*head_dim, hidden), wo (hidden,
 * n_heads*head_dim).  Supported: hidden and n_heads*head_dim in {1024, 2048},
 * and mep_attention's shapes.  h_out must not be h.
 *
 * mep_norm_head: logits (n_rows, vocab) fp32 = rms_norm(h + round(delta *
 * mult); norm) @ w^T / divisor for at most 32 rows, w (vocab, hidden) bf16,
 * hidden 1024 or 2048, products and sums in fp32 (modeling.py:249-254).
 * ---------------------------------------------------------------------- */
size_t mep_attention_block_workspace(int64_t n_rows, int32_t hidden, int32_t n_heads, int32_t n_kv_heads,
                                     int32_t head_dim);

int mep_attention_block(const void* h, const void* delta, float mult, const void* norm1, const void* norm2,
                        float eps, const void* wq, const void* wk, const void* wv, const void* wo,
                        const float* cos, const float* sin, int64_t n_positions, int32_t batch, int32_t t,
                        int32_t hidden, int32_t n_heads, int32_t n_kv_heads, int32_t head_dim, int64_t start,
                        int64_t max_len, float scale, float* k_cache, float* v_cache, void* workspace,
                        size_t workspace_bytes, void* h_out, void* x_out, void* stream);

int mep_norm_head(const void* h, const void* delta, float mult, const void* norm, float eps, const void* w,
                  int64_t n_rows, int32_t hidden, int32_t vocab, float divisor, float* logits, void* stream);

/* ------------------------------------------------------------------------
 * Projections of a bf16 model (modeling.py:160-185): out[i] (n_rows, cols[i])
 * = x (n_rows, k) @ w[i]^T for 1 to 3 matrices w[i] (cols[i], k) in one launch
 * (w, cols and out are host arrays of n_mats), fp32 sums rounded to bf16.
 * Supported: k a multiple of 128,
 * at least 256; cols multiples of 128; x and each matrix below 4 GiB.
 * ---------------------------------------------------------------------- */
int mep_linear(const void* x, int64_t n_rows, int32_t k, const void* const* w, const int32_t* cols,
               int32_t n_mats, void* const* out, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* MINIEP_AMD_MODEL_H */
