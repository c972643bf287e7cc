"""The model's linear layers under 16-bit autocast, with weight gradients from this build's kernel
(include/nanonemo_linear.h).

``projections(x, layers)`` applies bias-free ``nn.Linear`` layers that share an input: one product against their
stacked 16-bit weights, and in the backward one product for the input's gradient and one ``nn_linear_wgrad`` call for
every weight's, summed and returned in fp32. PyTorch's autocast runs a product per layer each way, rounds every weight
gradient to 16 bits and casts it back, and adds the input's gradients in 16 bits; the gradient products over
thousands of tokens into a small matrix are also where the library is slowest (768 x 768 over 8192 tokens: 50 us, of
which 10 would do).

``can_project(x, layers)`` says whether the call can take this path: plain CUDA tensors and untouched fp32
``nn.Linear`` layers under 16-bit autocast, in eager mode. Everything else (hooks, parametrizations, other module or
tensor types, torch.compile, torch.func, dispatch and function modes, forward-mode AD, no autocast, a stream capture with
gradients enabled) keeps calling the modules. A backward that is itself recorded (create_graph), or is handed gradients that the kernel cannot read by
address (is_grads_batched), runs differentiable torch products instead of the kernel.
"""

from __future__ import annotations

import torch
from torch import Tensor, nn
from torch.autograd import forward_ad
from torch.nn.modules import module as _module
from torch.utils._device import DeviceContext

from nanonemo_amd.kernels.hip import eager, host, records

_DTYPES = (torch.float16, torch.bfloat16)


def plain(m: nn.Module, x: Tensor, width: int, odd_rows: bool = False) -> bool:
    """Whether m is an untouched bias-free nn.Linear with an fp32 weight on x's device for inputs of this width
    (and of a multiple of 8 outputs, unless odd_rows)."""
    if type(m) is not nn.Linear or "forward" in m.__dict__:
        return False
    if m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks:
        return False
    own = m._parameters  # (read directly: a module's attribute lookup takes longer than the rest of this test)
    w = own.get("weight")
    if type(w) is not nn.Parameter or own.get("bias", m) is not None or w.dtype is not torch.float32 or w.device != x.device \
            or not w.is_contiguous():
        return False
    n, k = w.shape
    return (k == width and (odd_rows or n % 8 == 0) and k % 8 == 0 and n * k < 1 << 31  # the cast kernel's index, for four weights
            and w.data_ptr() % 16 == 0)


def function_mode() -> bool:
    """Whether a TorchFunctionMode is active that may intercept the modules' functions (torch.device's does not)."""
    n = torch._C._len_torch_function_stack()
    return n > 0 and any(type(torch._C._get_function_stack_at(i)) is not DeviceContext for i in range(n))


def eligible(x: Tensor) -> bool:
    """Whether a layer called on x now may run on this build's kernels (see above), whatever its modules."""
    if not eager(x) or not torch.is_autocast_enabled("cuda") or torch.get_autocast_dtype("cuda") not in _DTYPES:
        return False
    if x.dim() < 2 or x.numel() == 0 or not x.is_floating_point() or x.dtype is torch.float64:
        return False
    return not (torch.jit.is_tracing() or function_mode() or forward_ad._current_level >= 0 or _module._has_any_global_hook()
                or torch.is_grad_enabled() and torch.cuda.is_current_stream_capturing())


def can_project(x: Tensor, *layers: nn.Module) -> bool:
    """Whether ``projections`` can stand for calling the layers on x (see above)."""
    return eligible(x) and all(plain(m, x, x.shape[-1]) for m in layers)


def wgrad(dy: Tensor, x: Tensor, rows: list[int]) -> list[Tensor]:
    """dy^T x for dy (T, sum(rows)) and x (T, K), 16-bit with unit column strides: fp32, one (rows[i], K) tensor each."""
    return host().wgrad(dy, x, rows)


def stacked(grads: tuple[Tensor | None, ...], rows: list[int], like: Tensor) -> Tensor:
    """The gradients (T, rows[i]) side by side, zeros for an unused output."""
    if len(grads) == 1:
        return grads[0].contiguous()
    return torch.cat([like.new_zeros(like.shape[0], r) if g is None else g for g, r in zip(grads, rows)], dim=1)


class Stored(torch.autograd.Function):
    """The 16-bit copy that a forward made of a weight, as a function of the weight. A recorded backward computes with it:
    its derivatives reach the parameter, and its values are the forward's whatever has become of the parameter since
    (the nodes do not save the fp32 parameters, so changing one between forward and backward is no error, as with
    autocast's nn.Linear, which keeps the same copy)."""

    @staticmethod
    def forward(ctx, w, copy):
        return copy.detach()

    @staticmethod
    def backward(ctx, g):
        return g.float(), None


class _Projections(torch.autograd.Function):
    """y_i = x W_i^T: x (T, K) 16-bit, W_i fp32, y_i the column ranges of one (T, sum N_i) product."""

    @staticmethod
    def forward(ctx, x, turned, *ws):
        y, w16 = host().project_fwd(x, ws, turned)
        ctx.save_for_backward(x, w16)
        ctx.weights = ws
        ctx.set_materialize_grads(False)
        return (y,) if len(ws) == 1 else y.split([w.shape[0] for w in ws], dim=1)

    @staticmethod
    def backward(ctx, *dys):
        x, w16 = ctx.saved_tensors
        rows = [w.shape[0] for w in ctx.weights]
        need_w = any(ctx.needs_input_grad[2:])
        dy = stacked(dys, rows, x)
        if torch.is_grad_enabled() or not host().ordinary(dy):  # a recorded backward, or batched gradients
            wd = torch.cat([Stored.apply(w, c) for w, c in zip(ctx.weights, w16.split(rows))])
            dx = dy @ wd if ctx.needs_input_grad[0] else None
            dws = (dy.t() @ x).float().split(rows) if need_w else [None] * len(rows)
        else:
            dx = dy @ w16 if ctx.needs_input_grad[0] else None
            dws = wgrad(dy, x, rows) if need_w else [None] * len(rows)
        return dx, None, *(g if n else None for g, n in zip(dws, ctx.needs_input_grad[2:]))


def projections(x: Tensor, *layers: nn.Linear) -> tuple[Tensor, ...]:
    """The layers' outputs on x (..., K), in the autocast dtype, as (..., N_i) column ranges of one product."""
    flat = x.to(torch.get_autocast_dtype("cuda")).reshape(-1, x.shape[-1])
    return tuple(y.view(*x.shape[:-1], y.shape[1]) for y in _Projections.apply(flat, records(flat), *(m.weight for m in layers)))
