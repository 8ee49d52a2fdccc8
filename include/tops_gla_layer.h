/*
 * C entry points of libtops_gla.so that serve the GLA layer's decode step (tops.layers), beside
 * the kernel API of tops_gla.h, whose conventions they follow (device pointers, status codes,
 * the caller's stream; nothing is allocated and nothing synchronizes).
 */
#ifndef TOPS_GLA_LAYER_H
#define TOPS_GLA_LAYER_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/*
 * Bias-free projections of a few rows (decode steps), one launch: y_i [M, n_i] = x [M, K]
 * w_i^T for i < nw <= 8, weights w_i [n_i, K] bfloat16 row-major. x_dtype BF16: float32 sums
 * rounded once to bfloat16 (bit i of f32_mask: the rounded values stored as float32); F32:
 * float32 results at float32 accuracy. M <= 128, K a multiple of 256, every n_i a multiple of
 * 4, every pointer 16-byte aligned. Replaces the dense layers of tops/layers/gla.py:259-262,
 * 279-285, 333, 343 at decode sizes.
 */
int tops_gla_small_linear(const void* x, int x_dtype, const void* const* ws, const int64_t* ns,
                          int nw, int64_t M, int64_t K, void* const* ys, int f32_mask,
                          void* stream);

/*
 * The low-rank gate's second matrix with the gate: y [M, N] = max(log_sigmoid(x [M, R]
 * w [N, R]^T + bias [N]) / normalizer, clamp_min), bfloat16 throughout (the product plus bias
 * rounded to bfloat16 first); bias may be NULL, clamp only with has_clamp. R a multiple of 8.
 * Replaces tops/layers/gla.py:279-288 at decode sizes.
 */
int tops_gla_low_rank_gate(const void* x, const void* w, const void* bias, void* y, int64_t M,
                           int64_t N, int R, float normalizer, int has_clamp, float clamp_min,
                           void* stream);

#ifdef __cplusplus
}
#endif

#endif /* TOPS_GLA_LAYER_H */
