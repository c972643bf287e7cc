"""The model's output layer and loss as one call under 16-bit autocast: logits = x W^T and their mean cross entropy
(include/nanonemo_loss.h; /root/reference/nanonemo/model/model.py:60-66).

The loss reads the 16-bit logits once and its backward reads them once and writes their gradient, where F.cross_entropy
on logits.float() moves an fp32 copy, its log-softmax and their gradients. ``can_fuse_head`` holds for calls that
``linear.can_project`` describes with int64 targets; the others run module by module.
"""

from __future__ import annotations

import torch
import torch.nn.functional as F
from torch import Tensor, nn

from nanonemo_amd.kernels.hip import DTYPE_BF16, DTYPE_F16, check_loss, lib, on_device, stream_of
from nanonemo_amd.kernels.hip.linear import cast_weights, eligible, plain, wgrad

_DTYPES = {torch.float16: DTYPE_F16, torch.bfloat16: DTYPE_BF16}


def can_fuse_head(x: Tensor, layer: nn.Module, targets: Tensor) -> bool:
    """Whether ``head_loss`` can stand for F.cross_entropy(layer(x).float(), targets), rows flattened."""
    return (eligible(x) and x.dim() >= 2 and plain(layer, x, x.shape[-1], odd_rows=True) and type(targets) is Tensor
            and targets.dtype is torch.int64 and targets.device == x.device and targets.numel() == x.numel() // x.shape[-1]
            and not torch.cuda.is_current_stream_capturing())


class _HeadLoss(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w, targets):
        (w16,) = cast_weights(x.dtype, (w,))
        logits = x @ w16.t()
        R, V = logits.shape
        lse, rows, loss, inv = (torch.empty(n, dtype=torch.float32, device=x.device) for n in (R, R, (), ()))
        with on_device(x):
            check_loss(lib().nn_cross_entropy_fwd(logits.data_ptr(), targets.data_ptr(), lse.data_ptr(), rows.data_ptr(), loss.data_ptr(),
                                                  inv.data_ptr(), R, V, _DTYPES[x.dtype], stream_of(x)))
        ctx.save_for_backward(x, w16, w, targets, lse, inv)
        # The caller owns the logits and may change them in place before the backward, which then computes them again
        # from x: an alias that shares their version counter and not their graph, instead of a saved output, whose
        # change would be an error.
        ctx.logits = logits.detach()
        ctx.version = logits._version
        ctx.set_materialize_grads(False)
        return logits, loss

    @staticmethod
    def backward(ctx, dlogits, dloss):
        x, w16, w, targets, lse, inv = ctx.saved_tensors
        need_x, need_w, _ = ctx.needs_input_grad
        if torch.is_grad_enabled():
            return _replayed(x, w, targets, (need_x, need_w), dlogits, dloss)
        if dloss is not None:
            logits = ctx.logits if ctx.logits._version == ctx.version else x @ w16.t()
            d = torch.empty_like(logits)
            R, V = logits.shape
            dloss = dloss.contiguous()
            with on_device(x):
                check_loss(lib().nn_cross_entropy_bwd(logits.data_ptr(), targets.data_ptr(), lse.data_ptr(), inv.data_ptr(), dloss.data_ptr(),
                                                      d.data_ptr(), R, V, _DTYPES[x.dtype], stream_of(x)))
            dlogits = d if dlogits is None else d.add_(dlogits)
        if dlogits is None:
            return None, None, None
        dx = dlogits @ w16 if need_x else None
        dw = wgrad(dlogits.contiguous(), x, [w.shape[0]])[0] if need_w else None
        return dx, dw, None


def _replayed(x, w, targets, need, dlogits, dloss):
    """The gradients as recorded operations."""
    with torch.enable_grad():
        logits = F.linear(x, w.to(x.dtype))
        outs, grads = [], []
        if dlogits is not None:
            outs.append(logits), grads.append(dlogits)
        if dloss is not None:
            outs.append(F.cross_entropy(logits.float(), targets)), grads.append(dloss)
        if not outs:
            return None, None, None
        found = iter(torch.autograd.grad(outs, [t for t, n in zip((x, w), need) if n], grads, create_graph=True))
    return next(found) if need[0] else None, next(found) if need[1] else None, None


def head_loss(x: Tensor, layer: nn.Linear, targets: Tensor) -> tuple[Tensor, Tensor]:
    """(layer(x), the mean cross entropy of its rows against the targets) for calls that can_fuse_head."""
    flat = x.to(torch.get_autocast_dtype("cuda")).reshape(-1, x.shape[-1])
    logits, loss = _HeadLoss.apply(flat, layer.weight, targets.reshape(-1).contiguous())
    return logits.view(*x.shape[:-1], logits.shape[1]), loss
