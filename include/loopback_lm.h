/*
 * loopback_lm.h -- C ABI of libloopback_lm.so: the MI355X (gfx950) kernels of the language model around the Loopback
 * read (loopback_amd/lm.py) -- RMSNorm, SwiGLU and the next-token cross entropy, forward and backward, each one pass
 * over its rows; causal rotary attention in bf16 at head width 64, forward and backward; and the weight gradients of
 * bias-free linear layers in bf16. The reference leaves these to torch (looped_transformer.py:5-33, 431-615).
 *
 * Conventions: device pointers to contiguous row-major tensors; dtype is LDR_BF16 or LDR_F16 (loopback_read.h) for
 * the rows and weights, every statistic and partial sum is fp32, results are rounded once from fp32; stream is a
 * hipStream_t; nothing synchronizes with the host or allocates. The return value is 0, a negative code (rejected
 * before any launch: -1 argument, -2 shape, -3 alignment, -4 dtype) or a positive hipError_t.
 */
#ifndef LOOPBACK_LM_H
#define LOOPBACK_LM_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define LLM_ABI_VERSION 1
int llm_abi_version(void);

/* The widest row of llm_rms_norm_*: d a multiple of 8 up to this. */
#define LLM_NORM_MAX_WIDTH 2048

/* y = round(h r w), r = rsqrt(mean(h^2) + eps) into rstd [rows]; with add != NULL, h = round(x + add), stored to
 * h_out first (else h = x and h_out is not used). d a multiple of 8 up to LLM_NORM_MAX_WIDTH, rows 16-byte aligned. */
int llm_rms_norm_fwd(const void* x, const void* add, const void* w, void* h_out, void* y, float* rstd, int64_t rows,
                     int64_t d, float eps, int dtype, void* stream);

/* Rows of llm_rms_norm_bwd's weight-gradient partials. */
int64_t llm_rms_norm_parts(int64_t rows);

/* dx = round(r (dy w - h r mean(dy w h r)) + dres) (dres, another gradient of h, may be NULL) and the partial weight
 * gradients dw_part [llm_rms_norm_parts(rows), d], whose column sums are sum_rows dy h r. Either result may be NULL (not
 * wanted), not both. */
int llm_rms_norm_bwd(const void* dy, const void* h, const void* w, const float* rstd, const void* dres, void* dx,
                     float* dw_part, int64_t rows, int64_t d, int dtype, void* stream);

/* dw[c] = round(sum_p dw_part[p, c]) in a fixed order. */
int llm_sum_rows(const float* part, int64_t rows, int64_t d, void* out, int dtype, void* stream);

/* act = round(silu(g) u) for rows [g | u] of 2 n elements, n a multiple of 8; and its gradient d[g | u]. */
int llm_swiglu_fwd(const void* gate_up, void* act, int64_t rows, int64_t n, int dtype, void* stream);
int llm_swiglu_bwd(const void* gate_up, const void* dact, void* dgate_up, int64_t rows, int64_t n, int dtype,
                   void* stream);

/* Next-token cross entropy over logits [b, t, vocab] (element alignment) with labels ids[:, 1:], the last position of
 * each sequence ignored: lse [b t, 2] (each row's maximum and the log of its sum of exp(x - maximum)) and loss, the
 * mean over the b (t - 1) counted positions (fp32; NaN when there is none, or when an id is outside [0, vocab)).
 * scratch: b t floats. */
int llm_next_token_loss_fwd(const void* logits, const int64_t* ids, float* lse, float* scratch, float* loss, int64_t b,
                            int64_t t, int64_t vocab, int dtype, void* stream);

/* dlogits = round((softmax(logits) - onehot(label)) dloss / (b (t - 1))), zero rows at ignored positions. */
int llm_next_token_loss_bwd(const void* logits, const int64_t* ids, const float* lse, const float* dloss, void* dlogits,
                            int64_t b, int64_t t, int64_t vocab, int dtype, void* stream);

/* ---- causal rotary attention, head width 64, bf16 --------------------------------------------------------------
 * qkv [b, t, 3, heads, 64] (16-byte aligned); cos and sin [t, 64] fp32, both halves of a row alike. */

/* q and k rotated (pairs j, j + 32; x1 cos - x2 sin, x2 cos + x1 sin in fp32, one rounding) into qk [b, t, 2, heads,
 * 64]. */
int llm_rotary(const void* qkv, const float* cosT, const float* sinT, void* qk, int64_t b, int64_t t, int64_t heads,
               void* stream);

/* out [b, t, heads, 64] = softmax(q k^T / 8, causal) v from qk and qkv's v; lse2 [b heads, t], the base-2 logarithm of
 * each query's sum of exponentials, for the backward. */
int llm_attn_fwd(const void* qk, const void* qkv, void* out, float* lse2, int64_t b, int64_t t, int64_t heads,
                 void* stream);

/* dqkv [b, t, 3, heads, 64], the gradient of qkv through the rotation and the attention; delta: scratch [b heads, t]. */
int llm_attn_bwd(const void* qk, const void* qkv, const void* out, const void* dout, const float* lse2,
                 const float* cosT, const float* sinT, float* delta, void* dqkv, int64_t b, int64_t t, int64_t heads,
                 void* stream);

/* dw [n, k] = round(sum over m tokens of dy [m, n] x [m, k]), the weight gradient of a bias-free linear layer in bf16 (fp32
 * sums; n and k multiples of 8, 16-byte aligned). part: scratch, llm_wgrad_splits(m, n, k) x n x k floats. */
int64_t llm_wgrad_splits(int64_t m, int64_t n, int64_t k);
int llm_wgrad(const void* dy, const void* x, float* part, void* dw, int64_t m, int64_t n, int64_t k, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* LOOPBACK_LM_H */
