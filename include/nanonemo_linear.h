/* C ABI of the linear-layer kernels (gfx950): weight gradients, weight casts and the SwiGLU activation.
 * All pointers are device pointers; calls launch on `stream` and neither allocate nor synchronise. dtype: 0 fp16,
 * 1 bf16. Functions returning int give 0, or nonzero with nn_linear_last_error set. */
#ifndef NANONEMO_LINEAR_H
#define NANONEMO_LINEAR_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Weight gradient of y = x W^T: dW[n][k] = sum over t of dy[t][n] x[t][k], summed and stored in fp32. dy is [T][N]
 * with row stride ldy and x is [T][K] with row stride ldx (elements), both 16-bit; N, K and the strides are multiples
 * of 8 and the pointers 16-byte aligned. The N rows go to `nout` (1 to 3) dense outputs out[i] of rows[i] rows each
 * (sum of rows = N): the layers that share an input are one call. T = 0 writes zeros. Deterministic.
 * Replaces the bf16 product and the cast of autocast's nn.Linear backward (the projections of
 * /root/reference/nanonemo/model/layers.py:81-84,121-123). */
int nn_linear_wgrad(const void* dy, int64_t ldy, const void* x, int64_t ldx, int64_t T, int64_t N, int64_t K,
                    int nout, float* const* out, const int64_t* rows, void* workspace, size_t workspace_bytes,
                    int dtype, void* stream);

/* Bytes of workspace nn_linear_wgrad needs (16-byte aligned; 0 where it needs none). */
size_t nn_linear_wgrad_workspace_size(int64_t T, int64_t N, int64_t K);

/* dst[i] = src[i] rounded to the 16-bit dtype, for n (1 to 4) fp32 arrays of count[i] elements (multiples of 8,
 * 16-byte aligned), in one launch: a layer's weights at the start of its forward. */
int nn_linear_cast(int n, const float* const* src, void* const* dst, const int64_t* count, int dtype, void* stream);

/* The same for n (1 to 4) dense row-major matrices of rows[i] x cols[i] (multiples of 8), and each also transposed:
 * dst_t[i][c * ldt[i] + r] = dst[i][r * cols[i] + c], ldt[i] a multiple of 8, at least rows[i]. */
int nn_linear_cast_both(int n, const float* const* src, void* const* dst, void* const* dst_t, const int64_t* rows,
                        const int64_t* cols, const int64_t* ldt, int dtype, void* stream);

/* SwiGLU: h = silu(g) u with silu(g) = g / (1 + exp(-g)), in fp32 with one rounding. gu is [T][2 F] (a row's F values
 * of g, then its F values of u: the stacked product of the gate and up layers), h is [T][F]; dense, 16-byte aligned,
 * F a multiple of 8. The backward writes dgu = (dh u silu'(g), dh silu(g)), [T][2 F].
 * Replaces F.silu(gate) * up (/root/reference/nanonemo/model/layers.py:130-137). */
int nn_swiglu_fwd(const void* gu, void* h, int64_t T, int64_t F, int dtype, void* stream);
int nn_swiglu_bwd(const void* dh, const void* gu, void* dgu, int64_t T, int64_t F, int dtype, void* stream);

const char* nn_linear_last_error(void);

#ifdef __cplusplus
}
#endif

#endif /* NANONEMO_LINEAR_H */
