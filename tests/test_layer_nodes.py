"""CPU tests of the autograd nodes of the fused layers, output layer and projections (kernels/hip/layers.py, head.py,
linear.py) over a stand-in for the host module: what they accept, refuse, keep and release."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F
from torch import nn

from tests import host_standin


@pytest.fixture
def host(monkeypatch):
    return host_standin.install(monkeypatch)


def _head_inputs(V=24, d=16, R=10):
    torch.manual_seed(0)
    return nn.Linear(d, V, bias=False), torch.randn(R, d), torch.randint(0, V, (R,))


def test_head_loss_under_inference_mode(host):
    from nanonemo_amd.kernels.hip import head

    m, x, t = _head_inputs()
    with torch.no_grad():
        ref = head.head_loss(x, m, t)
    with torch.inference_mode():
        got = head.head_loss(x, m, t)
    assert all(torch.equal(a, b) for a, b in zip(got, ref))


def test_attention_layer_backward_refuses_capture(monkeypatch):
    # As the attention functions' backward does: a forward run eagerly and its backward under capture must not reach
    # the launches. The guard comes before the saved tensors are read.
    from nanonemo_amd.kernels.hip import layers

    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)

    class Ctx:
        needs_input_grad = (True,) * 12

        @property
        def saved_tensors(self):
            raise AssertionError("the guard must raise before the saved tensors are read")

    with pytest.raises(RuntimeError, match="attention layer backward: capturing"):
        layers._AttentionLayer.backward(Ctx(), torch.zeros(4, 8))


def test_head_loss_keeps_nothing_past_its_backward(host):
    # The logits are a saved tensor: autograd's hooks see them and a backward that does not retain the graph frees them,
    # while the caller may still change the logits it was given before the backward.
    from nanonemo_amd.kernels.hip import head

    m, x, t = _head_inputs()
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda v: packed.append(v) or v, lambda v: v):
        logits, loss = head.head_loss(x, m, t)
    assert logits.data_ptr() in [v.data_ptr() for v in packed]
    node = loss.grad_fn
    (g1,) = torch.autograd.grad(loss, m.weight, retain_graph=True)
    assert not host.recomputed
    with torch.no_grad():
        logits.mul_(2.0)
    (g2,) = torch.autograd.grad(loss, m.weight)
    assert host.recomputed
    torch.testing.assert_close(g1, g2)
    assert not any(isinstance(v, torch.Tensor) and v is not m.weight for v in vars(node).values())
    with pytest.raises(RuntimeError, match="freed"):
        node.saved_tensors


def _mlp(d=16, ff=24):
    torch.manual_seed(0)
    gate, up, down = nn.Linear(d, ff, bias=False), nn.Linear(d, ff, bias=False), nn.Linear(ff, d, bias=False)
    return torch.randn(3, 5, d, dtype=torch.bfloat16).requires_grad_(), (gate, up, down)


def _calls():
    """The fused calls: (output, its input, its layers)."""
    from nanonemo_amd.kernels.hip import head, layers, linear

    x, ws = _mlp()
    yield "mlp", lambda: layers.mlp_layer(x, *ws), x, ws
    yield "projections", lambda: torch.cat(linear.projections(x, *ws[:2]), -1), x, ws[:2]
    yield "projection", lambda: linear.projections(x, ws[0])[0], x, ws[:1]
    t = torch.randint(0, 24, (3, 5))
    yield "head", lambda: head.head_loss(x, ws[0], t)[1], x, ws[:1]


def test_weights_may_change_between_forward_and_backward(host):
    # As with autocast's nn.Linear, which keeps 16-bit copies: the backward, recorded or not, is the forward's.
    for name, f, x, ws in _calls():
        params = [m.weight for m in ws]
        ref = torch.autograd.grad(f().float().sum(), (x, *params))
        for recorded in (False, True):
            out, kept = f().float().sum(), [p.detach().clone() for p in params]
            with torch.no_grad():
                for p in params:
                    p.mul_(1.5)
            got = torch.autograd.grad(out, (x, *params), create_graph=recorded)
            with torch.no_grad():
                for p, k in zip(params, kept):
                    p.copy_(k)
            for a, b in zip(got, ref):
                torch.testing.assert_close(a, b, rtol=2e-2, atol=2e-2 * b.abs().max().item(), msg=f"{name} {recorded}")
            if recorded:  # and second derivatives reach the parameters
                assert any(g is not None for g in torch.autograd.grad(got[0].float().square().sum(), params, allow_unused=True)), name


def test_batched_gradients_pass_through_the_layers(host):
    # torch.autograd.grad(..., is_grads_batched=True) hands the backward tensors without storage of their own: they take
    # the replay, as they took the modules' backward.
    for name, f, x, ws in _calls():
        ins = (x, *(m.weight for m in ws))
        y = f()
        dys = torch.randn(4, *y.shape, dtype=y.dtype) if y.dim() else torch.tensor([0.5, -1.0, 2.0])
        got = torch.autograd.grad(y, ins, dys, is_grads_batched=True, retain_graph=True)
        for i, dy in enumerate(dys):
            for a, b in zip(got, torch.autograd.grad(y, ins, dy, retain_graph=True)):
                torch.testing.assert_close(a[i], b, rtol=2e-2, atol=2e-2 * b.abs().max().item(), msg=name)


def test_ordinary_tells_tensors_that_can_be_read_by_address():
    from nanonemo_amd.kernels.hip import host

    o = host().ordinary
    t = torch.randn(3, 4)
    assert o(t) and o(t.t()) and o(t.requires_grad_()) and o()
    assert not o(torch._efficientzerotensor(3)) and not o(torch.nested.nested_tensor([t.detach(), t.detach()])) and not o(t.detach().to_sparse())
    assert not o(torch.randn(3, dtype=torch.complex64).conj().imag) and not o(t, torch.randn(3, dtype=torch.complex64).conj())
    seen = []
    torch.func.vmap(lambda a: seen.append(o(a)) or a)(t.detach())
    torch.func.grad(lambda a: seen.append(o(a)) or a.sum())(t.detach())
    torch._vmap_internals._vmap(lambda a: seen.append(o(a)) or a, 0)(t.detach())
    assert seen == [False, False, False]


def test_function_modes_see_the_modules():
    # A TorchFunctionMode may replace F.linear or F.cross_entropy: the layers then run module by module. The mode behind
    # torch.set_default_device and `with torch.device(...)` replaces factories only.
    from nanonemo_amd.kernels.hip import linear

    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    assert not linear.function_mode()
    with torch.device("cpu"):
        assert not linear.function_mode()
        with Mode():
            assert linear.function_mode()
    with Mode():
        assert linear.function_mode()


def test_calls_past_the_kernels_indices_keep_the_modules(monkeypatch):
    # Sizes only (expanded tensors hold one value): no call that the modules answer may end in the library's refusal.
    from types import SimpleNamespace

    from nanonemo_amd.kernels import hip
    from nanonemo_amd.kernels.hip import head, host, layers, linear

    for m in (head, layers):
        monkeypatch.setattr(m, "eligible", lambda x: True)
        monkeypatch.setattr(m, "plain", lambda *_, **__: True)
    one = torch.zeros(1, dtype=torch.bfloat16)
    rows = lambda n, d: one.expand(n, d)  # noqa: E731
    for n, takes in (((1 << 24) - 1, True), (1 << 24, False)):  # a block per row, 2^32 threads in a launch
        assert head.can_fuse_head(rows(n, 8), None, torch.zeros(1, dtype=torch.int64).expand(n)) is takes
    assert hip.lib().nn_cross_entropy_fwd(*[None] * 6, 1 << 24, 8, 1, None) != 0 and b"invalid sizes" in hip.lib().nn_loss_last_error()
    H, KVH, hd, T = 12, 4, 64, 1024
    w = SimpleNamespace(weight=rows(H * hd, 64)), SimpleNamespace(weight=rows(KVH * hd, 64))
    cos = torch.zeros(T, hd // 2)
    for B, takes in (((1 << 31) // (T * (H + KVH) * (hd // 16)) - 1, True), ((1 << 31) // (T * (H + KVH) * (hd // 16)), False)):
        assert layers.can_fuse(one.expand(B, T, 64), cos, cos, H, KVH, hd, w[0], w[1], w[1], w[0]) is takes
    assert host().wgrad_takes((1 << 30) - 1, 8, 8) and not host().wgrad_takes(1 << 30, 8, 8)
    assert host().wgrad_takes(0, 8, 750000) and not host().wgrad_takes(64, 8, 750001) and not host().wgrad_takes(64, 12, 8)
    storage = torch.zeros(3 * (1 << 23) + 8, dtype=torch.bfloat16)
    near, far = (storage.as_strided((4, 8), (ld, 1)) for ld in ((1 << 23) - 8, 1 << 23))
    assert host().rows_aligned(near).data_ptr() == storage.data_ptr() and host().rows_aligned(far).is_contiguous()

    layer = nn.Linear(8, 8, bias=False)
    for n, takes in (((1 << 31) // 64 - 8, True), ((1 << 31) // 64, False)):
        layer.weight = nn.Parameter(torch.empty(n, 64, device="meta"))
        assert linear.plain(layer, torch.empty(1, device="meta"), 64) is takes


def test_stream_capture_with_gradients_keeps_the_modules(monkeypatch):
    # (without them the captured call is the eager one, and so are its results)
    from nanonemo_amd.kernels.hip import linear

    monkeypatch.setattr(linear, "eager", lambda *_: True)
    monkeypatch.setattr(torch, "is_autocast_enabled", lambda *_: True)
    monkeypatch.setattr(torch, "get_autocast_dtype", lambda *_: torch.bfloat16)
    m, x, _ = _head_inputs()
    for capturing in (False, True):
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
        assert linear.can_project(x, m) is not capturing
        with torch.no_grad():
            assert linear.can_project(x, m)
