/*
 * macko_decode.h -- C ABI of the glue kernels the batch-1 decode harness runs between the
 * matrix-vector products (libmacko_hip.so).  None of them has a counterpart in the upstream
 * package: its harness (python_scripts/util_run_pruned_llm.py:136-160) runs stock Hugging Face
 * modules for these parts.  They exist so that a decode step on MI355X is dominated by the
 * projections rather than by dozens of launch-bound framework kernels.
 *
 * All pointers are device pointers; activations fp16, tables fp32; `position` points at one
 * int64 in device memory (read by the kernel, so a captured graph can be replayed per token);
 * `stream` is a hipStream_t passed as void*.  Return codes as in macko_hip.h.
 */
#ifndef MACKO_DECODE_H
#define MACKO_DECODE_H

#include <stdint.h>

#include "macko_hip.h" /* MACKO_API, return codes */

#ifdef __cplusplus
extern "C" {
#endif

/* y[i] = x[i] * rsqrt(mean(x^2) + eps) * weight[i], i < n. */
MACKO_API int macko_decode_rmsnorm_f16(const void *x, const void *weight, void *y, int32_t n, float eps,
                             void *stream);

/*
 * Rotary embedding (rotate-half pairing: element i with i + head_dim/2) of q and k at
 * *position; writes the rotated q to q_out and appends the rotated k and v to the caches
 * [n_heads, max_len, head_dim] at that position.  cos_table / sin_table: [max_len, head_dim/2].
 */
MACKO_API int macko_decode_rope_append_f16(const void *q, const void *k, const void *v,
                                 const float *cos_table, const float *sin_table,
                                 const int64_t *position, void *q_out, void *k_cache,
                                 void *v_cache, int32_t n_heads, int32_t head_dim,
                                 int32_t max_len, void *stream);

/*
 * Single-query attention per head over cache positions 0..*position:
 * out = softmax(scale * q K^T) V.  head_dim <= 256 and a multiple of 8, max_len <= 4096,
 * both caches 16-byte aligned.
 */
MACKO_API int macko_decode_attention_f16(const void *q, const void *k_cache, const void *v_cache,
                               const int64_t *position, void *out, int32_t n_heads,
                               int32_t head_dim, int32_t max_len, float scale, void *stream);

/*
 * macko_decode_rope_append_f16 followed by macko_decode_attention_f16 in one launch: q, k, v are
 * the raw projections of the current token, the caches receive the rotated k and v at *position,
 * out is the attention output.  Same limits as the two separate calls.
 */
MACKO_API int macko_decode_rope_attention_f16(const void *q, const void *k, const void *v,
                                    const float *cos_table, const float *sin_table,
                                    const int64_t *position, void *k_cache, void *v_cache,
                                    void *out, int32_t n_heads, int32_t head_dim, int32_t max_len,
                                    float scale, void *stream);

/*
 * The same up to the last step: the context of every head is worked in MACKO_ATTENTION_PARTS pieces by
 * workgroups of their own, and their results are left as they are, to be merged by the product that
 * consumes them (macko_spmv_f16_attention_axpby).  head_dim 64 or 128, all pointers 16-byte aligned.
 *   parts  fp32 [n_heads][MACKO_ATTENTION_PARTS][head_dim], the sums of v weighted by exp(score - m_p),
 *          then [n_heads][MACKO_ATTENTION_PARTS][2], the pieces' (m_p, sum of the weights);
 *          out = sum_p exp(m_p - max m) parts_p / sum_p exp(m_p - max m) sum_p.
 */
#define MACKO_ATTENTION_PARTS 4
MACKO_API int macko_decode_rope_attention_parts_f16(const void *q, const void *k, const void *v,
                                          const float *cos_table, const float *sin_table,
                                          const int64_t *position, void *k_cache, void *v_cache,
                                          float *parts, int32_t n_heads, int32_t head_dim,
                                          int32_t max_len, float scale, void *stream);

/*
 * y [rows] = W rmsnorm(x) for a dense fp16 W [rows, cols], the normed vector rounded to fp16 in between (the output
 * layer of a decode step).  cols % 8 == 0, cols <= 4096; w, x and norm_weight 16-byte aligned.
 */
MACKO_API int macko_decode_norm_matvec_f16(const void *w, const void *x, const void *norm_weight, void *y,
                                 int32_t rows, int32_t cols, float eps, void *stream);

/* out[i] = silu(gate[i]) * up[i], i < n. */
MACKO_API int macko_decode_silu_mul_f16(const void *gate, const void *up, void *out, int32_t n,
                              void *stream);

/*
 * The same parts for all tokens of a prompt at once.  Rows are contiguous, every pointer is 16-byte
 * aligned, cols % 8 == 0; `packed` is written in the operand order of macko_spmv_f16_packed
 * (macko_packed_bytes(cols, batch) bytes).
 *   pack_rmsnorm   packed = rmsnorm(x[b, :]) * weight
 *   pack_silu_mul  packed = silu(gate[b, :]) * up[b, :]
 *   rope_append    q [batch, n_heads * head_dim] rotated in place, k rotated and v into the caches
 *                  [n_heads, max_len, head_dim] at positions[b]; cos_rows / sin_rows fp16
 *                  [batch, head_dim], both halves of a row alike; head_dim % 16 == 0
 *   attention      packed = attention of token b over cache positions 0..positions[b]; q rotated,
 *                  head_dim 64 or 128
 */
MACKO_API int macko_prefill_pack_rmsnorm_f16(const void *x, const void *weight, void *packed, int32_t cols,
                                   int32_t batch, float eps, void *stream);
/* y[b, :] = rmsnorm(x[b, :]) * weight as plain rows. */
MACKO_API int macko_rmsnorm_rows_f16(const void *x, const void *weight, void *y, int32_t cols,
                           int32_t batch, float eps, void *stream);
MACKO_API int macko_prefill_pack_silu_mul_f16(const void *gate, const void *up, void *packed, int32_t cols,
                                    int32_t batch, void *stream);
MACKO_API int macko_prefill_rope_append_f16(void *q, const void *k, const void *v, const void *cos_rows,
                                  const void *sin_rows, const int64_t *positions, void *k_cache,
                                  void *v_cache, int32_t batch, int32_t n_heads, int32_t head_dim,
                                  int32_t max_len, void *stream);
MACKO_API int macko_prefill_attention_f16(const void *q, const void *k_cache, const void *v_cache,
                                const int64_t *positions, void *packed, int32_t batch,
                                int32_t n_heads, int32_t head_dim, int32_t max_len, float scale,
                                void *stream);

#ifdef __cplusplus
}
#endif
#endif /* MACKO_DECODE_H */
