"""The model's attention layer and MLP as one call each under 16-bit autocast, forward and backward
(/root/reference/nanonemo/model/layers.py:77-116,119-137).

Attention: projections, rotary embedding, attention and output projection. The layer's own memory order lets every
kernel read what the one before it wrote: q, k and v are column ranges of one product's (B T, (H + 2 KVH) hd) output, the
rotation writes q to a tensor of its own and k over itself, the attention reads k and v where they lie (nn_fa_fwd_views),
and the backward writes dq, dk and dv as column ranges of one buffer, rotates them back in place and hands it to one
product for the input's gradient and one call for the three weights'.
That is 6 launches forward and 9 to 11 backward, where the modules take 27 in all: a cast, a product and a rounding
per weight each way, three input gradients added in 16 bits.

MLP: one product for gate and up, SwiGLU on its two halves (nn_swiglu_*), the down product; backward, one call for
the gate's and up's weight gradients and one product for the input's gradient. 4 launches forward and 6 to 8 backward
instead of 21.

A layer's weights are rounded to 16 bits in one launch at the start of its forward; where a backward will be run
(``turned``), a transposed copy is written beside them, which the products for the inputs' gradients read.

``can_fuse`` and ``can_fuse_mlp`` hold for the calls that ``linear.can_project`` describes, with every module of the layer
untouched; the others run module by module. A backward that is itself recorded, or is handed gradients that the kernels
cannot read by address (is_grads_batched), replays the layer through PyTorch's linear layers and the package's
differentiable functions, so that what those support is what it supports.
"""

from __future__ import annotations

import torch
import torch.nn.functional as F
from torch import Tensor, nn

from nanonemo_amd.kernels.hip import host, records
from nanonemo_amd.kernels.hip.flash_attn import _refuse_capture_with_autograd, flash_attn_bthd
from nanonemo_amd.kernels.hip.linear import Stored, eligible, plain
from nanonemo_amd.kernels.hip.rope import rope_qk


def can_fuse(x: Tensor, cos: Tensor, sin: Tensor, heads: int, kv_heads: int, hd: int, wq, wk, wv, wo) -> bool:
    """Whether ``attention_layer`` can stand for the layer's modules called on x."""
    if not eligible(x) or x.dim() != 3 or hd not in (32, 64):
        return False
    B, T, d = x.shape
    if not (plain(wq, x, d) and plain(wk, x, d) and plain(wv, x, d) and plain(wo, x, heads * hd)):
        return False
    # the library's row offsets within a sequence, and the rotation kernel's index
    if T * (heads + 2 * kv_heads) * hd >= 1 << 30 or B * T * (heads + kv_heads) * (hd // 16) >= 1 << 31:
        return False
    if wq.weight.shape[0] != heads * hd or wk.weight.shape[0] != kv_heads * hd or wv.weight.shape[0] != kv_heads * hd:
        return False
    for t in (cos, sin):
        if type(t) is not Tensor or t.dtype is not torch.float32 or t.device != x.device or t.requires_grad \
                or t.dim() != 2 or t.shape[0] < T or t.shape[1] != hd // 2 or not t.is_contiguous():
            return False
    return True


class _AttentionLayer(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, cos, sin, B, T, H, KVH, wq, wk, wv, wo, turned):
        y, qkv, q, o, lse, w, wo16 = host().attention_layer_fwd(x, cos, sin, B, T, H, KVH, wq, wk, wv, wo, turned)
        ctx.save_for_backward(x, cos, sin, qkv, q, o, lse, w, wo16)
        ctx.weights, ctx.sizes = (wq, wk, wv, wo), (B, T, H, KVH)
        return y

    @staticmethod
    def backward(ctx, dy):
        _refuse_capture_with_autograd("attention layer backward")
        x, cos, sin, qkv, q, o, lse, w, wo16 = ctx.saved_tensors
        need = ctx.needs_input_grad
        if torch.is_grad_enabled() or not host().ordinary(dy):
            copies = (*w.split([m.shape[0] for m in ctx.weights[:3]]), wo16)
            dx, *dws = _replayed(_modular, x, ctx.weights, copies, (need[0], *need[7:11]), dy, (cos, sin, *ctx.sizes))
            return dx, None, None, None, None, None, None, *dws, None
        dx, *dws = host().attention_layer_bwd(dy, x, cos, sin, qkv, q, o, lse, w, wo16, *ctx.sizes, need[0], any(need[7:10]), need[10])
        return dx, None, None, None, None, None, None, *(g if n else None for g, n in zip(dws, need[7:11])), None


def _modular(x, wq, wk, wv, wo, cos, sin, B, T, H, KVH):
    """The layer through differentiable functions, on (B T, d) x and weights of x's dtype."""
    D = wq.shape[0] // H
    q, k, v = (F.linear(x, w).view(B, T, -1, D) for w in (wq, wk, wv))
    q, k = rope_qk(q, k, cos, sin)
    return F.linear(flash_attn_bthd(q, k, v).view(B * T, H * D), wo)


def _replayed(fn, x, weights, copies, need, dy, extra=()) -> list:
    """The gradients of fn(x, *weights, *extra) as torch operations, recorded if the backward is, on the forward's 16-bit
    copies of the weights."""
    record = torch.is_grad_enabled()
    with torch.enable_grad():
        y = fn(x, *(Stored.apply(w, c) for w, c in zip(weights, copies)), *extra)
        grads = iter(torch.autograd.grad(y, [t for t, n in zip((x, *weights), need) if n], dy, create_graph=record))
    return [next(grads) if n else None for n in need]


def attention_layer(x: Tensor, cos: Tensor, sin: Tensor, heads: int, kv_heads: int, wq: nn.Linear, wk: nn.Linear,
                    wv: nn.Linear, wo: nn.Linear) -> Tensor:
    """wo(attention(rope(wq x), rope(wk x), wv x)) on x (B, T, d) in the autocast dtype, for calls that can_fuse."""
    B, T, d = x.shape
    flat = x.to(torch.get_autocast_dtype("cuda")).reshape(B * T, d)
    y = _AttentionLayer.apply(flat, cos, sin, B, T, heads, kv_heads, wq.weight, wk.weight, wv.weight, wo.weight,
                              records(flat, wq.weight, wk.weight, wv.weight))
    return y.view(B, T, -1)


def can_fuse_mlp(x: Tensor, w_gate, w_up, w_down) -> bool:
    """Whether ``mlp_layer`` can stand for the MLP's modules called on x."""
    if not eligible(x) or x.dim() < 2:
        return False
    d = x.shape[-1]
    if not (plain(w_gate, x, d) and plain(w_up, x, d)):
        return False
    F_ = w_gate.weight.shape[0]
    return (w_up.weight.shape[0] == F_ and plain(w_down, x, F_) and x.numel() // d * F_ < 1 << 33)  # the activation kernel's index


class _MlpLayer(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w_gate, w_up, w_down, turned):
        y, gu, h, w, wd = host().mlp_fwd(x, w_gate, w_up, w_down, turned)
        ctx.save_for_backward(x, gu, h, w, wd)
        ctx.weights = (w_gate, w_up, w_down)
        return y

    @staticmethod
    def backward(ctx, dy):
        x, gu, h, w, wd = ctx.saved_tensors
        need = ctx.needs_input_grad[:4]
        if torch.is_grad_enabled() or not host().ordinary(dy):
            return *_replayed(_modular_mlp, x, ctx.weights, (*w.chunk(2), wd), need, dy), None
        grads = host().mlp_bwd(dy, x, gu, h, w, wd, need[0], need[1] or need[2], need[3])
        return *(g if n else None for g, n in zip(grads, need)), None


def _modular_mlp(x, w_gate, w_up, w_down):
    """The MLP through differentiable functions, on weights of x's dtype."""
    return F.linear(F.silu(F.linear(x, w_gate)) * F.linear(x, w_up), w_down)


def mlp_layer(x: Tensor, w_gate: nn.Linear, w_up: nn.Linear, w_down: nn.Linear) -> Tensor:
    """w_down(silu(w_gate x) * w_up x) on x (..., d) in the autocast dtype, for calls that can_fuse_mlp."""
    flat = x.to(torch.get_autocast_dtype("cuda")).reshape(-1, x.shape[-1])
    y = _MlpLayer.apply(flat, w_gate.weight, w_up.weight, w_down.weight, records(flat, w_gate.weight, w_up.weight))
    return y.view(*x.shape[:-1], y.shape[1])
