"""torch.library op for the gfx950 RoPE kernel (include/nanonemo_rope.h): q and k rotated in one launch.

Replaces the reference's RoPE on either side of the attention op: the plain-PyTorch apply_rope
(/root/reference/nanonemo/model/layers.py:67-74, upcast, two muls and an add per half, a cat and a
downcast per tensor) and its fused Triton apply_rope_qk (nanonemo/kernels/triton/rope.py, used at
layers.py:99-101), which rotates q and k in the (B, T, heads, hd) projection layout in one launch.

    rope_qk(q, k, cos, sin) -> (q', k')      q (B, T, H, hd), k (B, T, KVH, hd); cos/sin fp32 (T_max, hd/2)

The result is bit-identical to the reference's torch formula (fp32 products and sums rounded one at a
time, then one rounding to the input dtype), and so is the gradient (the rotation by -theta).
"""

from __future__ import annotations

import torch
from torch import Tensor
from torch.autograd.function import once_differentiable

from nanonemo_amd.kernels.hip import eager, host, preload, records


@torch.library.custom_op("nanonemo::rope_qk", mutates_args=())
def _rope_qk(q: Tensor, k: Tensor, cos: Tensor, sin: Tensor) -> tuple[Tensor, Tensor]:
    return host().rope(q, k, cos, sin, False)


@_rope_qk.register_fake
def _(q, k, cos, sin):
    return torch.empty(q.shape, dtype=q.dtype, device=q.device), torch.empty(k.shape, dtype=k.dtype, device=k.device)


@torch.library.custom_op("nanonemo::rope_qk_bwd", mutates_args=())
def _rope_qk_bwd(dq: Tensor, dk: Tensor, cos: Tensor, sin: Tensor) -> tuple[Tensor, Tensor]:
    return host().rope(dq, dk, cos, sin, True)


@_rope_qk_bwd.register_fake
def _(dq, dk, cos, sin):
    return torch.empty(dq.shape, dtype=dq.dtype, device=dq.device), torch.empty(dk.shape, dtype=dk.dtype, device=dk.device)


def _setup_context(ctx, inputs, output):
    _, _, cos, sin = inputs
    ctx.save_for_backward(cos, sin)


def _backward(ctx, dq, dk):
    cos, sin = ctx.saved_tensors
    gq, gk = _rope_qk_bwd(dq, dk, cos, sin)
    return gq, gk, None, None


_rope_qk.register_autograd(_backward, setup_context=_setup_context)


class _RopeQkFn(torch.autograd.Function):
    """The eager path of rope_qk (plain CUDA tensors outside tracing; ``eager``): the op's launches and autograd
    wiring without its dispatch, so the same bits for less host time."""

    @staticmethod
    def forward(ctx, q, k, cos, sin):
        ctx.save_for_backward(cos, sin)
        return host().rope(q, k, cos, sin, False)

    @staticmethod
    @once_differentiable
    def backward(ctx, dq, dk):
        cos, sin = ctx.saved_tensors
        gq, gk = host().rope(dq, dk, cos, sin, True)
        return gq, gk, None, None


def _rope(q: Tensor, k: Tensor, cos: Tensor, sin: Tensor) -> tuple[Tensor, Tensor]:
    if eager(q, k, cos, sin):
        if records(q, k, cos, sin):
            return _RopeQkFn.apply(q, k, cos, sin)
        return host().rope(q, k, cos, sin, False)
    return _rope_qk(q, k, cos, sin)


def rope_qk(q: Tensor, k: Tensor, cos: Tensor, sin: Tensor) -> tuple[Tensor, Tensor]:
    """Rotate q (B, T, H, hd) and k (B, T, KVH, hd) by the positions' angles (cos/sin: fp32 (T_max, hd/2))."""
    return _rope(q, k, cos, sin)


def rope_k(k: Tensor, cos: Tensor, sin: Tensor) -> Tensor:
    """Rotate k (B, T, KVH, hd) alone (the q half of the pass is folded into the attention op)."""
    q = k.new_empty(k.shape[0], k.shape[1], 0, k.shape[3])
    return _rope(q, k, cos, sin)[1]


preload()
