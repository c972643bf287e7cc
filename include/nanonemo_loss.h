/* C ABI of the cross-entropy kernels (gfx950). All pointers are device pointers; calls launch on `stream` and neither
 * allocate nor synchronise. dtype: 0 fp16, 1 bf16, 2 fp32. Functions returning int give 0, or nonzero with
 * nn_loss_last_error set.
 * Replaces F.cross_entropy on fp32 logits (/root/reference/nanonemo/model/model.py:62-66): the mean over the rows whose
 * target is not -100 of logsumexp(row) - row[target], in fp32; NaN where no row counts, or a target is out of range. */
#ifndef NANONEMO_LOSS_H
#define NANONEMO_LOSS_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* logits: [R][V] dense, R < 2^24; targets: int64 [R]. Writes lse[R] (logsumexp, fp32), rows[R] (scratch: the rows' losses),
 * loss[1] and inv[1] = 1 / number of rows that count. Deterministic. */
int nn_cross_entropy_fwd(const void* logits, const int64_t* targets, float* lse, float* rows, float* loss, float* inv,
                         int64_t R, int64_t V, int dtype, void* stream);

/* dlogits = (softmax(logits) - onehot(target)) * grad[0] * inv[0], zero for rows that do not count (NaN if their logits
 * hold a NaN or +inf, as in PyTorch); lse and inv as the
 * forward wrote them, grad the gradient of the loss (one fp32), dlogits in the logits' dtype. NaN in a row whose target is
 * out of range. */
int nn_cross_entropy_bwd(const void* logits, const int64_t* targets, const float* lse, const float* inv,
                         const float* grad, void* dlogits, int64_t R, int64_t V, int dtype, void* stream);

const char* nn_loss_last_error(void);

#ifdef __cplusplus
}
#endif

#endif /* NANONEMO_LOSS_H */
