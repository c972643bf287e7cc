"""The model's output layer and loss as one call under 16-bit autocast: logits = x W^T and their mean cross entropy
(include/nanonemo_loss.h; /root/reference/nanonemo/model/model.py:60-66).

The loss reads the 16-bit logits once and its backward reads them once and writes their gradient, where F.cross_entropy
on logits.float() moves an fp32 copy, its log-softmax and their gradients. ``can_fuse_head`` holds for calls that
``linear.can_project`` describes with int64 targets; the others run module by module. A target that is neither -100 nor in
[0, V) makes the loss and its row's gradient NaN (F.cross_entropy ends the process with a device assertion).
"""

from __future__ import annotations

import torch
import torch.nn.functional as F
from torch import Tensor, nn

from nanonemo_amd.kernels.hip import host, records
from nanonemo_amd.kernels.hip.linear import Stored, eligible, plain


def can_fuse_head(x: Tensor, layer: nn.Module, targets: Tensor) -> bool:
    """Whether ``head_loss`` can stand for F.cross_entropy(layer(x).float(), targets), rows flattened."""
    return (eligible(x) and x.dim() >= 2 and plain(layer, x, x.shape[-1], odd_rows=True) and type(targets) is Tensor
            and targets.dtype is torch.int64 and targets.device == x.device and targets.numel() == x.numel() // x.shape[-1]
            and targets.numel() < 1 << 24)  # a block per row, and a launch ends at 2^32 threads


class _HeadLoss(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w, targets, turned):
        logits, loss, w16, lse, inv = host().head_fwd(x, w, targets, turned)
        # The caller owns the logits and may change them in place before the backward, which then computes them again
        # from x. Saved is an alias with a version of its own (saving the output would make such a change an error);
        # whether the logits have changed is read from their own version, which holds on to no memory.
        ctx.save_for_backward(x, w16, targets, lse, inv, logits.data)
        ctx.weight, ctx.version, ctx.at = w, host().Version(logits), logits._version
        ctx.set_materialize_grads(False)
        return logits, loss

    @staticmethod
    def backward(ctx, dlogits, dloss):
        x, w16, targets, lse, inv, logits = ctx.saved_tensors
        need_x, need_w = ctx.needs_input_grad[:2]
        if torch.is_grad_enabled() or not host().ordinary(*(g for g in (dlogits, dloss) if g is not None)):
            return *_replayed(x, ctx.weight, w16, targets, (need_x, need_w), dlogits, dloss), None
        if ctx.version.current() != ctx.at:
            logits = None
        return (*host().head_bwd(dlogits, dloss, logits, x, w16, targets, lse, inv, need_x, need_w), None, None)


def _replayed(x, w, w16, targets, need, dlogits, dloss):
    """The gradients as torch operations, recorded if the backward is, on the forward's 16-bit copy of the weight."""
    record = torch.is_grad_enabled()
    with torch.enable_grad():
        logits = F.linear(x, Stored.apply(w, w16))
        outs, grads = [], []
        if dlogits is not None:
            outs.append(logits), grads.append(dlogits)
        if dloss is not None:
            outs.append(F.cross_entropy(logits.float(), targets)), grads.append(dloss)
        if not outs:
            return None, None, None
        found = iter(torch.autograd.grad(outs, [t for t, n in zip((x, w), need) if n], grads, create_graph=record))
    return next(found) if need[0] else None, next(found) if need[1] else None, None


def head_loss(x: Tensor, layer: nn.Linear, targets: Tensor) -> tuple[Tensor, Tensor]:
    """(layer(x), the mean cross entropy of its rows against the targets) for calls that can_fuse_head."""
    flat = x.to(torch.get_autocast_dtype("cuda")).reshape(-1, x.shape[-1])
    targets = targets.reshape(-1).contiguous()
    if records(flat, layer.weight):
        logits, loss = _HeadLoss.apply(flat, layer.weight, targets, records(flat))
    else:  # nothing to keep for a backward (inference tensors have no version to keep either)
        logits, loss = host().head_fwd(flat, layer.weight, targets, False)[:2]
    return logits.view(*x.shape[:-1], logits.shape[1]), loss
