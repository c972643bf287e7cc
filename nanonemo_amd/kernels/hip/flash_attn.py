"""torch.library boundary of the gfx950 causal GQA FlashAttention-2 kernels.

Drop-in for /root/reference/nanonemo/kernels/cuda/flash_attn.py: the same op names and schemas
(``nanonemo::flash_attn`` :18-22 and ``nanonemo::flash_attn_bwd`` :31-35), the same fake impls
(contiguous outputs, :25-28 and :38-40), the same autograd wiring (save q, k, v, o, lse; ignore the
gradient of lse, :43-54) and the same public ``flash_attn(q, k, v) -> o`` (:57-60). Under
``torch.compile(fullgraph=True)`` each op is one opaque node traced through its fake impl.

Differences from the reference, all widening: fp16 **and** bf16 inputs (the reference accepts fp16
only, flash_attn.cu:344-346), and the compute is the HIP library behind a C ABI
(include/nanonemo_fa.h) called by the host module (csrc/host.cpp) on PyTorch's current HIP stream. Every
output and the backward workspace is allocated there by PyTorch's caching allocator; the library never
allocates, synchronises or copies to the host, so both ops can be captured into a HIP graph. On CUDA tensors
the ops' kernels are the host module's (the bodies here serve other devices, which they refuse). In eager
mode the public functions reach the same launches through a plain autograd.Function instead of the ops'
dispatch (see "the eager path" below).
"""

from __future__ import annotations

import torch
from torch import Tensor
from torch.autograd.function import once_differentiable

from nanonemo_amd.kernels.hip import eager as _eager
from nanonemo_amd.kernels.hip import host, preload
from nanonemo_amd.kernels.hip import records as _records


def _contig(t: Tensor) -> Tensor:
    return t if t.is_contiguous() else t.contiguous()


_CAPTURE_MSG = (
    "{}: capturing this op into a HIP graph while autograd records it (torch.cuda.graph around the forward and its "
    "autograd backward, or torch.compile(mode='reduce-overhead')) is not supported: such a capture once ended in a "
    "host fault in capture_end and no cause has been shown. Capture the C ABI calls (nn_fa_fwd / nn_fa_bwd / "
    "nn_fa_bwd_noalloc) instead, or run the ops eagerly (torch.compile(fullgraph=True) without graphs is supported)."
)


def _refuse_capture_with_autograd(where: str, *inputs: Tensor) -> None:
    """Raise when the current stream is capturing and autograd will record this op: before any launch in the
    public functions (grad mode on and an input requires grad), and in setup_context / the backward as a
    backstop for direct op calls. Capture without autograd, and capture of the C ABI, are unaffected. Skipped
    while torch.compile traces (the check is a host query, and no capture runs at trace time)."""
    # A capture needs PyTorch's initialised HIP state: is_initialized is a flag read, where the capture query is a
    # runtime call, and this runs on every op call.
    if inputs and not (torch.is_grad_enabled() and any(t.requires_grad for t in inputs)):
        return
    if not torch.cuda.is_initialized():
        return
    if torch.compiler.is_compiling() or not torch.cuda.is_current_stream_capturing():
        return
    raise RuntimeError(_CAPTURE_MSG.format(where))


@torch.library.custom_op("nanonemo::flash_attn", mutates_args=())
def _flash_attn(q: Tensor, k: Tensor, v: Tensor) -> tuple[Tensor, Tensor]:
    return host().fa_fwd(q, k, v)


@_flash_attn.register_fake
def _(q, k, v):
    B, H, T, _ = q.shape  # the kernel returns contiguous tensors whatever the input strides
    return (
        torch.empty(q.shape, dtype=q.dtype, device=q.device),
        torch.empty((B, H, T), dtype=torch.float32, device=q.device),
    )


@torch.library.custom_op("nanonemo::flash_attn_bwd", mutates_args=())
def _flash_attn_bwd(d_o: Tensor, q: Tensor, k: Tensor, v: Tensor, o: Tensor, lse: Tensor) -> tuple[Tensor, Tensor, Tensor]:
    return host().fa_bwd_op(d_o, q, k, v, o, lse)


@_flash_attn_bwd.register_fake
def _(d_o, q, k, v, o, lse):
    return tuple(torch.empty(t.shape, dtype=t.dtype, device=t.device) for t in (q, k, v))


def _setup_context(ctx, inputs, output):
    _refuse_capture_with_autograd("flash_attn (autograd)")
    q, k, v = inputs
    o, lse = output
    ctx.save_for_backward(q, k, v, o, lse)
    # lse's gradient is ignored, so autograd need not fill a zero tensor for it on every backward.
    ctx.set_materialize_grads(False)


def _d_out(d_o, o):
    """The gradient reaching o; zeros when o itself was not used (only lse was), as a materialised grad would be."""
    return torch.zeros_like(o) if d_o is None else d_o


def _backward(ctx, d_o, _d_lse):
    _refuse_capture_with_autograd("flash_attn backward")
    q, k, v, o, lse = ctx.saved_tensors
    return _flash_attn_bwd(_d_out(d_o, o), q, k, v, o, lse)


_flash_attn.register_autograd(_backward, setup_context=_setup_context)


# ---- the eager path of the public functions ----------------------------------------------------
# The custom ops are what torch.compile traces (one opaque node each, through their fake impls) and what callers
# of torch.ops.nanonemo.* reach. Run eagerly under autograd, an op pays for the dispatcher's Python kernel, the
# autograd.Function that register_autograd generates and, in the backward, a second op's dispatch and checks: tens
# of microseconds of host time per forward + backward, which at the model's shape is about the GPU time of the
# three kernels. The public functions therefore run plain CUDA tensors in eager mode through the
# autograd.Functions below (``eager``): the same checks and launches in the forward, and in the backward the
# launch alone, on the inputs the forward checked and saved (the gradient autograd hands over has o's
# shape and dtype). Outputs and gradients are the same bits as the ops'. Everything else (torch.compile tracing,
# torch.func transforms, dispatch modes, tensor subclasses, meta and CPU tensors) goes through the custom ops.


class _FlashAttnFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v):
        if not (q.is_contiguous() and k.is_contiguous() and v.is_contiguous()):  # copies the backward would make again
            (q,), (k, v) = host().readable(q), host().readable(k, v)
        o, lse = host().fa_fwd(q, k, v)
        ctx.save_for_backward(q, k, v, o, lse)
        ctx.set_materialize_grads(False)
        return o

    @staticmethod
    @once_differentiable
    def backward(ctx, d_o):
        _refuse_capture_with_autograd("flash_attn backward")
        q, k, v, o, lse = ctx.saved_tensors
        return host().fa_bwd(_d_out(d_o, o), q, k, v, o, lse)


def flash_attn(q: Tensor, k: Tensor, v: Tensor) -> Tensor:
    """Causal GQA attention. q: (B, H, T, hd), k/v: (B, KVH, T, hd), fp16 or bf16, H % KVH == 0, hd in {32, 64}."""
    _refuse_capture_with_autograd("flash_attn", q, k, v)
    if _eager(q, k, v):
        return _FlashAttnFn.apply(q, k, v) if _records(q, k, v) else host().fa_fwd(q, k, v)[0]
    o, _ = _flash_attn(q, k, v)
    return o


# ---- layout-fused ops: (B, T, heads, hd) in and out -------------------------------------------
# The reference model projects x to (B, T, heads * hd), views it as (B, T, heads, hd), transposes to
# (B, heads, T, hd) for the op (which then copies each input to contiguous memory,
# /root/reference/nanonemo/kernels/cuda/flash_attn.py:20,33) and transposes + reshapes o back for
# the output projection (/root/reference/nanonemo/model/layers.py:97-104,116), one more copy per
# direction. These ops take and return the projection layout itself through the library's strided
# entry points: q (B, T, H, hd), k / v (B, T, KVH, hd), o / dq (B, T, H, hd), dk / dv (B, T, KVH, hd),
# all contiguous in that layout (so o.view(B, T, H * hd) feeds the output projection directly);
# lse stays (B, H, T). Not in the reference: an addition that the same model code can select.


@torch.library.custom_op("nanonemo::flash_attn_bthd", mutates_args=())
def _flash_attn_bthd(q: Tensor, k: Tensor, v: Tensor) -> tuple[Tensor, Tensor]:
    return host().bthd_fwd(q, k, v)


@_flash_attn_bthd.register_fake
def _(q, k, v):
    B, T, H, _ = q.shape
    return (
        torch.empty(q.shape, dtype=q.dtype, device=q.device),
        torch.empty((B, H, T), dtype=torch.float32, device=q.device),
    )


@torch.library.custom_op("nanonemo::flash_attn_bthd_bwd", mutates_args=())
def _flash_attn_bthd_bwd(
    d_o: Tensor, q: Tensor, k: Tensor, v: Tensor, o: Tensor, lse: Tensor
) -> tuple[Tensor, Tensor, Tensor]:
    return host().bthd_bwd_op(d_o, q, k, v, o, lse)


@_flash_attn_bthd_bwd.register_fake
def _(d_o, q, k, v, o, lse):
    return tuple(torch.empty(t.shape, dtype=t.dtype, device=t.device) for t in (q, k, v))


def _backward_bthd(ctx, d_o, _d_lse):
    _refuse_capture_with_autograd("flash_attn_bthd backward")
    q, k, v, o, lse = ctx.saved_tensors
    return _flash_attn_bthd_bwd(_d_out(d_o, o), q, k, v, o, lse)


_flash_attn_bthd.register_autograd(_backward_bthd, setup_context=_setup_context)


class _FlashAttnBthdFn(torch.autograd.Function):
    """The eager path of flash_attn_bthd (see flash_attn's)."""

    @staticmethod
    def forward(ctx, q, k, v):
        q, k, v = _contig(q), _contig(k), _contig(v)
        o, lse = host().bthd_fwd(q, k, v)
        ctx.save_for_backward(q, k, v, o, lse)
        ctx.set_materialize_grads(False)
        return o

    @staticmethod
    @once_differentiable
    def backward(ctx, d_o):
        _refuse_capture_with_autograd("flash_attn_bthd backward")
        q, k, v, o, lse = ctx.saved_tensors
        return host().bthd_bwd(_d_out(d_o, o), q, k, v, o, lse)


def flash_attn_bthd(q: Tensor, k: Tensor, v: Tensor) -> Tensor:
    """Causal GQA attention in the projection layout: q (B, T, H, hd), k/v (B, T, KVH, hd) -> o (B, T, H, hd)."""
    _refuse_capture_with_autograd("flash_attn_bthd", q, k, v)
    if _eager(q, k, v):
        if _records(q, k, v):
            return _FlashAttnBthdFn.apply(q, k, v)
        return host().bthd_fwd(q, k, v)[0]
    o, _ = _flash_attn_bthd(q, k, v)
    return o


# ---- RoPE of q folded into the layout-fused ops ------------------------------------------------
# The reference rotates q and k beside the op (/root/reference/nanonemo/model/layers.py:99-101) and the op
# then reads the rotated tensors. Here the forward takes q *before* RoPE, rotates each query row in registers
# (the same fp32 operation order as nanonemo::rope_qk, so the result is bit-identical) and also returns the
# rotated q, which the backward reads; the backward's dQ kernel rotates its gradient back by -theta before
# storing it, so dq is the gradient of the unrotated q. k is rotated beforehand (rope_k). Not in the reference:
# an addition the same model code can select (rope_kernel="fused"). The gradients of lse and of the rotated q
# output are not propagated (the model uses neither), as the reference ignores lse's.


@torch.library.custom_op("nanonemo::flash_attn_bthd_rope", mutates_args=())
def _flash_attn_bthd_rope(q: Tensor, k: Tensor, v: Tensor, cos: Tensor, sin: Tensor) -> tuple[Tensor, Tensor, Tensor]:
    return host().bthd_rope_fwd(q, k, v, cos, sin)


@_flash_attn_bthd_rope.register_fake
def _(q, k, v, cos, sin):
    B, T, H, _ = q.shape
    return (
        torch.empty(q.shape, dtype=q.dtype, device=q.device),
        torch.empty((B, H, T), dtype=torch.float32, device=q.device),
        torch.empty(q.shape, dtype=q.dtype, device=q.device),
    )


@torch.library.custom_op("nanonemo::flash_attn_bthd_rope_bwd", mutates_args=())
def _flash_attn_bthd_rope_bwd(
    d_o: Tensor, q_rot: Tensor, k: Tensor, v: Tensor, o: Tensor, lse: Tensor, cos: Tensor, sin: Tensor
) -> tuple[Tensor, Tensor, Tensor]:
    return host().bthd_rope_bwd_op(d_o, q_rot, k, v, o, lse, cos, sin)


@_flash_attn_bthd_rope_bwd.register_fake
def _(d_o, q_rot, k, v, o, lse, cos, sin):
    return tuple(torch.empty(t.shape, dtype=t.dtype, device=t.device) for t in (q_rot, k, v))


def _setup_context_rope(ctx, inputs, output):
    _refuse_capture_with_autograd("flash_attn_bthd_rope (autograd)")
    _, k, v, cos, sin = inputs
    o, lse, q_rot = output
    ctx.save_for_backward(q_rot, k, v, o, lse, cos, sin)
    ctx.set_materialize_grads(False)  # the gradients of lse and q_rot are ignored


def _backward_rope(ctx, d_o, _d_lse, _d_q_rot):
    _refuse_capture_with_autograd("flash_attn_bthd_rope backward")
    q_rot, k, v, o, lse, cos, sin = ctx.saved_tensors
    dq, dk, dv = _flash_attn_bthd_rope_bwd(_d_out(d_o, o), q_rot, k, v, o, lse, cos, sin)
    return dq, dk, dv, None, None


_flash_attn_bthd_rope.register_autograd(_backward_rope, setup_context=_setup_context_rope)


class _FlashAttnBthdRopeFn(torch.autograd.Function):
    """The eager path of flash_attn_bthd_rope (see flash_attn's)."""

    @staticmethod
    def forward(ctx, q, k, v, cos, sin):
        k, v = _contig(k), _contig(v)
        o, lse, q_rot = host().bthd_rope_fwd(q, k, v, cos, sin)
        ctx.save_for_backward(q_rot, k, v, o, lse, cos, sin)
        ctx.set_materialize_grads(False)
        return o

    @staticmethod
    @once_differentiable
    def backward(ctx, d_o):
        _refuse_capture_with_autograd("flash_attn_bthd_rope backward")
        q_rot, k, v, o, lse, cos, sin = ctx.saved_tensors
        dq, dk, dv = host().bthd_rope_bwd(_d_out(d_o, o), q_rot, k, v, o, lse, cos, sin)
        return dq, dk, dv, None, None


def flash_attn_bthd_rope(q: Tensor, k: Tensor, v: Tensor, cos: Tensor, sin: Tensor) -> Tensor:
    """Causal GQA attention in the projection layout with q's RoPE folded in: q (B, T, H, hd) *before* RoPE,
    k (B, T, KVH, hd) already rotated, v (B, T, KVH, hd), cos/sin fp32 (T_max, hd/2) -> o (B, T, H, hd)."""
    _refuse_capture_with_autograd("flash_attn_bthd_rope", q, k, v)
    if _eager(q, k, v, cos, sin):
        if _records(q, k, v, cos, sin):
            return _FlashAttnBthdRopeFn.apply(q, k, v, cos, sin)
        return host().bthd_rope_fwd(q, k, v, cos, sin)[0]
    o, _, _ = _flash_attn_bthd_rope(q, k, v, cos, sin)
    return o


preload()
