/*
 * crane_few.h -- C ABI of the projections of a decode step of one sequence
 * (gfx950): candle Linear (qwen3/modeling.rs:382-387, 466, 573-591),
 * optionally with the residual add and RmsNorm, or decode attention, in front of it
 * (qwen3/modeling.rs:655-673) or SiLU(gate) * up behind it
 * (crane-core/src/fused_ops) in the same launch.  Results and roundings are
 * those of crane_hip_add_rms_norm (or crane_hip_rms_norm), crane_gemm_linear and
 * crane_hip_silu_mul one after the other; the f32 sums associate in the kernel's
 * own order.  Conventions as in crane_hip.h; nothing allocates, synchronises or
 * needs a workspace.
 */
#ifndef CRANE_FEW_H
#define CRANE_FEW_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* 1 when the calls below take the shape, else 0: bf16, M = 1, K a multiple of
 * 512 up to 4096 with the norm, to 32768 without.  N rows of weight; gated: N = 2
 * inter. */
int crane_few_supported(int64_t M, int64_t N, int64_t K, int norm, int gated, int dtype);

/* y[M, N] = x[M, K] w[N, K]^T (+ bias[N] or NULL). */
int crane_few_linear(const void* x, const void* w, const void* bias, void* y, int64_t M, int64_t N, int64_t K,
                     int dtype, void* stream);

/* residual = T(x + hidden) and h = RmsNorm(residual, norm_w), or without hidden
 * (NULL) h = RmsNorm(x, norm_w) and residual is not written (may be NULL); then
 * y[M, N] = h w^T (+ bias), or with gated y[M, N / 2] = silu(g) * u, [g | u] =
 * T(h w^T) (no bias).  x, hidden, residual [M, K]; residual is not x or hidden. */
int crane_few_norm_linear(const void* x, const void* hidden, const void* norm_w, void* residual, float eps,
                          const void* w, const void* bias, void* y, int64_t M, int64_t N, int64_t K, int gated,
                          int dtype, void* stream);

/* 1 when crane_few_attn_linear takes the sizes, else 0: bf16, 256 < max_kv <=
 * 2048, N <= 1024, Hq a multiple of 4 up to 16. */
int crane_few_attn_linear_supported(int64_t max_kv, int Hq, int64_t N, int dtype);

/* y[1, N] = attention w[N, Hq D]^T: crane_hip_attn_decode of one sequence and
 * crane_few_linear (o_proj), with the merge of the attention's partials inside
 * the product.  Arguments as crane_hip_attn_decode with B = 1; attn: scratch for
 * the attention row [Hq D] (its contents are unspecified afterwards). */
int crane_few_attn_linear(const void* q, const void* k_cache, const void* v_cache, int64_t cache_cap,
                          const int32_t* kv_len, int64_t max_kv, int Hq, int Hkv, int D, float scale, int score_mode,
                          void* workspace, size_t ws_bytes, void* attn, const void* w, void* y, int64_t N, int dtype,
                          void* stream);

#ifdef __cplusplus
}
#endif
#endif /* CRANE_FEW_H */
