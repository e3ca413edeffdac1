/*
 * tfgfa_gpt2.h - C ABI of the GPT-2 block kernels around the attention (MI355X, gfx950).
 *
 * The reference's block runs its norms, GELU, residual adds and the one-token projections as
 * separate PyTorch operators (src/py/model_inference.py:39-164).  These entry points compute
 * the same functions in one pass each.  Values are float32 with float32 arithmetic; a result
 * marked bf16 is rounded once, to nearest even.
 *
 * Conventions as in tfgfa.h: device pointers, the caller owns every buffer, launches are
 * asynchronous on `hip_stream`, arguments are checked before any HIP call; 0 on success, > 0
 * an invalid argument (TFGFA_ERR_*; TFGFA_ERR_TOO_LARGE past one launch's threads), < 0 a negated
 * hipError_t.  Tensors are contiguous and 16-byte
 * aligned.  Row counts of 0 launch nothing.
 */
#ifndef TFGFA_GPT2_H
#define TFGFA_GPT2_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Largest row width of the norm (a row lives in one wave's registers), the most rows of the
 * few-row projections (8 normed rows of 1600 take 50 of the 60 KiB of LDS they may; more rows were
 * not measured) and the most arrays of one cast. */
#define TFGPT2_MAX_NORM_DIM 2048
#define TFGPT2_MAX_ROWS     8
#define TFGPT2_MAX_CASTS    10
/* One launch takes fewer than 2^32 threads: the most rows of a norm (a wave each), values of a GELU or of
 * one call's casts (four a thread), outputs of a few-row projection with a norm (64 threads an output). */
#define TFGPT2_MAX_NORM_ROWS 67108863LL
#define TFGPT2_MAX_VALUES    17179868160LL
#define TFGPT2_MAX_OUTPUTS   67108860
/* Most splits of the contraction of tfgpt2_linear_planes. */
#define TFGPT2_MAX_K_SPLITS 8

/* What a result is written as.  PLANES: (3, rows, width) bf16, three arrays whose values add up to
 * the float32 result exactly (where it is infinite or NaN: itself, then NaN). */
#define TFGPT2_F32    0
#define TFGPT2_BF16   1
#define TFGPT2_PLANES 2

/*
 * LayerNorm over rows of width d (a multiple of 4, at most TFGPT2_MAX_NORM_DIM), biased variance:
 *   s = x            (delta == NULL)
 *   s = x + delta    (delta: (rows, d) bf16; s is also written to sum, (rows, d) float32)
 *   y = (s - mean) / sqrt(var + eps) * scale + shift
 * y is (rows, d), as y_kind says.  sum may be x itself.
 * src/py/model_inference.py:96-107 (LayerNorm), :157-160 (the residual add before norm2).
 */
int tfgpt2_layernorm(const float* x, const void* delta, float* sum, const float* scale,
                     const float* shift, void* y, int y_kind, int64_t rows, int d, float eps,
                     void* hip_stream);

/*
 * GELU, tanh form, elementwise over n float32 values:
 *   y = 0.5 x (1 + tanh(sqrt(2 / pi) (x + 0.044715 x^3)))      (model_inference.py:109-117)
 */
int tfgpt2_gelu(const float* x, float* y, int64_t n, void* hip_stream);

/*
 * float32 -> bf16 copies of up to TFGPT2_MAX_CASTS arrays in one launch: dst[i][0 .. n[i]) = src[i][0 .. n[i]).
 * n[i] a multiple of 4.
 */
int tfgpt2_cast_bf16(int count, const float* const* src, void* const* dst, const int64_t* n,
                     void* hip_stream);

/*
 * A linear layer on few rows (1 <= M <= TFGPT2_MAX_ROWS), the projections of one decode step:
 *   y[m, n] = f( sum_k xhat[m, k] w[n, k] + bias[n] ) + residual[m, n]
 * with up to three weight matrices sharing x (query, key and value): parts in 1..3, part p uses
 * w[p] (N, K) float32, bias[p] (N) float32 or NULL, y[p] (M, N).
 *   x        (M, K), float32 (x_bf16 = 0) or bf16 (x_bf16 = 1)
 *   ln_scale, ln_shift   both NULL, or (K): xhat = LayerNorm(x) with eps, as above (x float32,
 *                        K <= TFGPT2_MAX_NORM_DIM, M * (K + 4) <= 15360); otherwise xhat = x
 *   gelu     1: f is the GELU above (with a norm, float32 y), 0: identity
 *   residual (M, N) float32 or NULL (parts == 1); y[0] may be residual itself
 *   y_bf16   element type of every y: float32 (0), or bf16 (1) with a norm and no GELU
 * K a multiple of 4.  Products and sums are float32; the result does not depend on the device or
 * the launch.
 */
int tfgpt2_linear_rows(const void* x, int x_bf16, const float* ln_scale, const float* ln_shift,
                       float eps, int parts, const float* const* w, const float* const* bias,
                       int gelu, const float* residual, void* const* y, int y_bf16, int M, int N,
                       int K, void* hip_stream);

/*
 * A float32 linear layer on the bf16 matrix units:
 *   y = x w^T + bias (+ residual)          (M, N) float32          gelu_planes = 0
 *   y = GELU(x w^T + bias) as PLANES       (3, M, N) bf16          gelu_planes = 1 (no residual)
 *   x  (3, M, K) bf16 PLANES    w  (N, K) float32    bias  (N) or NULL    residual  (M, N) or NULL
 * Every product is that of the float32 values to 2^-26 of itself, sums are float32: as close to the
 * exact result as a float32 GEMM.  A sum that is not finite is computed again from float32 products, so
 * infinities, NaN and overflow give what they give there.  An operand below 2^-103 in magnitude is
 * taken to an absolute 2^-125: its lower pieces leave bf16's normal range.
 * splits: 1..TFGPT2_MAX_K_SPLITS partial sums of the contraction, tfgpt2_linear_planes_splits' choice
 * for a device of cu_count CUs (0: sizes not taken: N a multiple of 4, K of 32, planes and weights
 * below 2 GiB).  part: splits * M * N floats (NULL for one split); the partial sums are
 * added in order, so the result depends on the sizes and `splits` only.
 */
int tfgpt2_linear_planes_splits(int M, int N, int K, int cu_count);
int tfgpt2_linear_planes(const void* x, const float* w, const float* bias, int gelu_planes,
                         const float* residual, void* y, float* part, int splits, int M, int N,
                         int K, void* hip_stream);

#ifdef __cplusplus
}
#endif

#endif /* TFGFA_GPT2_H */
