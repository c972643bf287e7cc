"""The model's attention layer and MLP as one call each under 16-bit autocast, forward and backward
(/root/reference/nanonemo/model/layers.py:77-116,119-137).

Attention: projections, rotary embedding, attention and output projection. The layer's own memory order lets every kernel read what the one before it wrote: q, k and v are column ranges of one
product's (B T, (H + 2 KVH) hd) output, the rotation writes q to a tensor of its own and k over itself, the attention
reads k and v where they lie (nn_fa_fwd_views), and the backward writes dq, dk and dv as column ranges of one buffer,
rotates them back in place and hands it to one product for the input's gradient and one call for the three weights'.
That is 6 launches forward and 9 to 11 backward, where the modules take 27 in all: a cast, a product and a rounding
per weight each way, three input gradients added in 16 bits.

MLP: one product for gate and up, SwiGLU on its two halves (nn_swiglu_*), the down product; backward, one call for
the gate's and up's weight gradients and one product for the input's gradient. 4 launches forward and 6 to 8 backward
instead of 21.

``can_fuse`` and ``can_fuse_mlp`` hold for the calls that ``linear.can_project`` describes, with every module of the layer untouched; the others run module by module. A backward that is itself recorded replays the layer through PyTorch's linear layers
and the package's differentiable functions, so that what those support is what it supports.
"""

from __future__ import annotations

import ctypes
import math

import torch
import torch.nn.functional as F
from torch import Tensor, nn

from nanonemo_amd.kernels.hip import DTYPE_BF16, DTYPE_F16, check, check_linear, check_rope, lib, on_device, stream_of
from nanonemo_amd.kernels.hip.flash_attn import flash_attn_bthd
from nanonemo_amd.kernels.hip.linear import cast_weights, eligible, plain, wgrad
from nanonemo_amd.kernels.hip.rope import rope_qk

_DTYPES = {torch.float16: DTYPE_F16, torch.bfloat16: DTYPE_BF16}


def can_fuse(x: Tensor, cos: Tensor, sin: Tensor, heads: int, kv_heads: int, hd: int, wq, wk, wv, wo) -> bool:
    """Whether ``attention_layer`` can stand for the layer's modules called on x."""
    if not eligible(x) or x.dim() != 3 or hd not in (32, 64):
        return False
    d = x.shape[2]
    if not (plain(wq, x, d) and plain(wk, x, d) and plain(wv, x, d) and plain(wo, x, heads * hd)):
        return False
    if wq.weight.shape[0] != heads * hd or wk.weight.shape[0] != kv_heads * hd or wv.weight.shape[0] != kv_heads * hd:
        return False
    for t in (cos, sin):
        if type(t) is not Tensor or t.dtype is not torch.float32 or t.device != x.device or t.requires_grad \
                or t.dim() != 2 or t.shape[0] < x.shape[1] or t.shape[1] != hd // 2 or not t.is_contiguous():
            return False
    return not torch.cuda.is_current_stream_capturing()


class _Shape:
    """Sizes of a call, and the strides of its tensors for the library."""

    def __init__(self, B: int, T: int, H: int, KVH: int, D: int):
        self.B, self.T, self.H, self.KVH, self.D = B, T, H, KVH, D
        self.nq, self.nk = H * D, KVH * D
        n = self.n = self.nq + 2 * self.nk
        dense, wide = (T * self.nq, D, self.nq), (T * n, D, n)  # {batch, head, row}: q, o and dO; ranges of the buffer
        self.fwd = (ctypes.c_int64 * 9)(*dense, *wide, *dense)
        self.bwd = (ctypes.c_int64 * 15)(*dense, *wide, *dense, *wide, *wide)
        dense_r, wide_r = (dense[0], dense[2], D), (wide[0], wide[2], D)  # {batch, position, head}
        self.rot = (ctypes.c_int64 * 12)(*wide_r, *dense_r, *wide_r, *wide_r)
        self.unrot = (ctypes.c_int64 * 12)(*wide_r * 4)

    def ranges(self, buf: Tensor) -> tuple[int, int, int]:
        """Addresses of the q, k and v ranges of a (B T, n) buffer."""
        p = buf.data_ptr()
        return p, p + 2 * self.nq, p + 2 * (self.nq + self.nk)


class _AttentionLayer(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, cos, sin, B, T, H, KVH, wq, wk, wv, wo):
        sh = _Shape(B, T, H, KVH, wq.shape[0] // H)
        w, wo16 = cast_weights(x.dtype, (wq, wk, wv), (wo,))
        qkv = x @ w.t()
        q_rot = torch.empty((B, T, sh.nq), dtype=x.dtype, device=x.device)
        o = torch.empty_like(q_rot)
        lse = torch.empty((B, H, T), dtype=torch.float32, device=x.device)
        L, dt, D = lib(), _DTYPES[x.dtype], sh.D
        q, k, v = sh.ranges(qkv)
        with on_device(x):
            st = stream_of(x)
            check_rope(L.nn_rope_qk_views(q, q_rot.data_ptr(), k, k, cos.data_ptr(), sin.data_ptr(), B, T, H, KVH, D, sh.rot,
                                          cos.shape[0], dt, 0, st))
            check(L.nn_fa_fwd_views(q_rot.data_ptr(), k, v, o.data_ptr(), lse.data_ptr(), B, H, KVH, T, D, sh.fwd, dt,
                                    1.0 / math.sqrt(D), st))
        y = o.view(B * T, sh.nq) @ wo16.t()
        ctx.save_for_backward(x, cos, sin, qkv, q_rot, o, lse, w, wo16, wq, wk, wv, wo)
        ctx.sh = sh
        return y

    @staticmethod
    def backward(ctx, dy):
        x, cos, sin, qkv, q_rot, o, lse, w, wo16, wq, wk, wv, wo = ctx.saved_tensors
        sh, need = ctx.sh, ctx.needs_input_grad
        B, T, H, KVH, D = sh.B, sh.T, sh.H, sh.KVH, sh.D
        if torch.is_grad_enabled():
            return _replayed(_modular, (x, wq, wk, wv, wo), (need[0], *need[7:]), dy, (cos, sin, B, T, H, KVH), at=7)
        dy = dy.contiguous()
        d_o = dy @ wo16
        dwo = wgrad(dy, o.view(B * T, sh.nq), [wo.shape[0]])[0] if need[10] else None
        if not (need[0] or any(need[7:10])):
            return None, None, None, None, None, None, None, None, None, None, dwo
        dqkv = torch.empty_like(qkv)
        L, dt = lib(), _DTYPES[x.dtype]
        ws_bytes = L.nn_fa_bwd_workspace_size(B, H, KVH, T, D)
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device=x.device)
        _, k, v = sh.ranges(qkv)
        dq, dk, dv = sh.ranges(dqkv)
        with on_device(x):
            st = stream_of(x)
            check(L.nn_fa_bwd_views(d_o.data_ptr(), q_rot.data_ptr(), k, v, o.data_ptr(), lse.data_ptr(), dq, dk, dv,
                                    ws.data_ptr(), ws_bytes, B, H, KVH, T, D, sh.bwd, dt, 1.0 / math.sqrt(D), st))
            check_rope(L.nn_rope_qk_views(dq, dq, dk, dk, cos.data_ptr(), sin.data_ptr(), B, T, H, KVH, D, sh.unrot,
                                          cos.shape[0], dt, 1, st))
        dx = dqkv @ w if need[0] else None
        dws = wgrad(dqkv, x, [sh.nq, sh.nk, sh.nk]) if any(need[7:10]) else [None] * 3
        return dx, None, None, None, None, None, None, *(g if n else None for g, n in zip(dws, need[7:10])), dwo


def _modular(x, wq, wk, wv, wo, cos, sin, B, T, H, KVH):
    """The layer through differentiable functions, on (B T, d) x, in x's dtype."""
    D = wq.shape[0] // H
    q, k, v = (F.linear(x, w.to(x.dtype)).view(B, T, -1, D) for w in (wq, wk, wv))
    q, k = rope_qk(q, k, cos, sin)
    return F.linear(flash_attn_bthd(q, k, v).view(B * T, H * D), wo.to(x.dtype))


def _replayed(fn, ins, need, dy, extra, at: int) -> tuple:
    """The gradients of fn(*ins, *extra) as recorded operations: x's first, then None up to position ``at``, then the
    weights'."""
    with torch.enable_grad():
        y = fn(*ins, *extra)
        grads = iter(torch.autograd.grad(y, [t for t, n in zip(ins, need) if n], dy, create_graph=True))
    out = [next(grads) if n else None for n in need]
    return (out[0], *[None] * (at - 1), *out[1:])


def attention_layer(x: Tensor, cos: Tensor, sin: Tensor, heads: int, kv_heads: int, wq: nn.Linear, wk: nn.Linear,
                    wv: nn.Linear, wo: nn.Linear) -> Tensor:
    """wo(attention(rope(wq x), rope(wk x), wv x)) on x (B, T, d) in the autocast dtype, for calls that can_fuse."""
    B, T, d = x.shape
    flat = x.to(torch.get_autocast_dtype("cuda")).reshape(B * T, d)
    y = _AttentionLayer.apply(flat, cos, sin, B, T, heads, kv_heads, wq.weight, wk.weight, wv.weight, wo.weight)
    return y.view(B, T, -1)


def can_fuse_mlp(x: Tensor, w_gate, w_up, w_down) -> bool:
    """Whether ``mlp_layer`` can stand for the MLP's modules called on x."""
    if not eligible(x) or x.dim() < 2:
        return False
    d = x.shape[-1]
    if not (plain(w_gate, x, d) and plain(w_up, x, d)):
        return False
    F_ = w_gate.weight.shape[0]
    return w_up.weight.shape[0] == F_ and plain(w_down, x, F_) and not torch.cuda.is_current_stream_capturing()


class _MlpLayer(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w_gate, w_up, w_down):
        wgu, wd = cast_weights(x.dtype, (w_gate, w_up), (w_down,))
        gu = x @ wgu.t()
        T, F_ = x.shape[0], w_gate.shape[0]
        h = torch.empty((T, F_), dtype=x.dtype, device=x.device)
        with on_device(x):
            check_linear(lib().nn_swiglu_fwd(gu.data_ptr(), h.data_ptr(), T, F_, _DTYPES[x.dtype], stream_of(x)))
        y = h @ wd.t()
        ctx.save_for_backward(x, gu, h, wgu, wd, w_gate, w_up, w_down)
        return y

    @staticmethod
    def backward(ctx, dy):
        x, gu, h, wgu, wd, w_gate, w_up, w_down = ctx.saved_tensors
        need = ctx.needs_input_grad
        if torch.is_grad_enabled():
            return _replayed(_modular_mlp, (x, w_gate, w_up, w_down), need, dy, (), at=1)
        dy = dy.contiguous()
        dwd = wgrad(dy, h, [w_down.shape[0]])[0] if need[3] else None
        if not (need[0] or need[1] or need[2]):
            return None, None, None, dwd
        dh = dy @ wd
        dgu = torch.empty_like(gu)
        T, F_ = h.shape
        with on_device(x):
            check_linear(lib().nn_swiglu_bwd(dh.data_ptr(), gu.data_ptr(), dgu.data_ptr(), T, F_, _DTYPES[x.dtype], stream_of(x)))
        dx = dgu @ wgu if need[0] else None
        dwg, dwu = wgrad(dgu, x, [F_, F_]) if need[1] or need[2] else (None, None)
        return dx, dwg if need[1] else None, dwu if need[2] else None, dwd


def _modular_mlp(x, w_gate, w_up, w_down):
    """The MLP through differentiable functions, in x's dtype."""
    return F.linear(F.silu(F.linear(x, w_gate.to(x.dtype))) * F.linear(x, w_up.to(x.dtype)), w_down.to(x.dtype))


def mlp_layer(x: Tensor, w_gate: nn.Linear, w_up: nn.Linear, w_down: nn.Linear) -> Tensor:
    """w_down(silu(w_gate x) * w_up x) on x (..., d) in the autocast dtype, for calls that can_fuse_mlp."""
    flat = x.to(torch.get_autocast_dtype("cuda")).reshape(-1, x.shape[-1])
    y = _MlpLayer.apply(flat, w_gate.weight, w_up.weight, w_down.weight)
    return y.view(*x.shape[:-1], y.shape[1])
