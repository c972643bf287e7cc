"""GPU tests of the fused layers (kernels/hip/layers.py) against the same modules run one by one and against float64."""

from __future__ import annotations

import copy

import pytest
import torch

from nanonemo_amd.model import MLP, Attention, ModelConfig, rope_tables

pytestmark = pytest.mark.gpu


def _attention(H, KVH, hd, T, **kw):
    torch.manual_seed(0)
    cfg = ModelConfig(n_layers=1, d_model=H * hd, n_heads=H, n_kv_heads=KVH, max_seq_len=T, attn_kernel="hip_bthd", **kw)
    return Attention(cfg).cuda(), tuple(t.cuda() for t in rope_tables(hd, T, 10000.0))


def _modules_only(m):
    """The same module with a no-op hook on each linear layer, which keeps every call on the modules."""
    m = copy.copy(m)
    m._modules = {n: copy.deepcopy(c) for n, c in m._modules.items()}
    for c in m._modules.values():
        c.register_forward_hook(lambda *_: None)
    return m


def _run(m, args, dy, dtype):
    with torch.autocast("cuda", dtype=dtype):
        y = m(*args)
    return (y.detach(), *torch.autograd.grad(y, (args[0], *m.parameters()), dy))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
# From T = 3: at T = 1 the softmax is constant and the exact gradients of wq and wk are 0, so two correct results differ
# by all of their rounding noise.
@pytest.mark.parametrize("B, T, H, KVH, hd", [(2, 200, 12, 4, 64), (1, 3, 4, 1, 32), (3, 65, 2, 2, 64), (1, 1030, 8, 2, 32)])
def test_attention_layer_matches_its_modules(B, T, H, KVH, hd, dtype):
    from nanonemo_amd.kernels.hip import layers

    print(f"\n[case] attention layer B={B} T={T} H={H} KVH={KVH} hd={hd} {dtype}", flush=True)
    m, (cos, sin) = _attention(H, KVH, hd, T, rope_kernel="hip")
    x = torch.randn(B, T, H * hd, device="cuda").to(dtype).requires_grad_()
    dy = torch.randn(B, T, H * hd, device="cuda").to(dtype)
    ref_m = _modules_only(m)
    with torch.autocast("cuda", dtype=dtype):
        assert layers.can_fuse(x, cos, sin, H, KVH, hd, m.wq, m.wk, m.wv, m.wo)
        assert not layers.can_fuse(x, cos, sin, H, KVH, hd, ref_m.wq, ref_m.wk, ref_m.wv, ref_m.wo)
    got, ref = _run(m, (x, cos, sin), dy, dtype), _run(ref_m, (x, cos, sin), dy, dtype)
    # the same 16-bit products with other sums; the reference rounds weight gradients and partial input gradients too
    tol = 2e-2 if dtype == torch.bfloat16 else 3e-3
    for name, a, b in zip(("y", "dx", "dwq", "dwk", "dwv", "dwo"), got, ref):
        assert a.shape == b.shape and a.dtype == b.dtype, name
        torch.testing.assert_close(a, b, rtol=tol, atol=tol * b.abs().max().item(), msg=name)
    with torch.no_grad(), torch.autocast("cuda", dtype=dtype):
        assert torch.equal(m(x, cos, sin), got[0])


def _rel(a, b):
    """The 2-norm of a - b over b's, in float64."""
    return ((a.double() - b).norm() / b.norm()).item()


def _attention64(x, cos, sin, H, KVH, wq, wk, wv, wo):
    B, T, _ = x.shape
    c, s = cos[:T, None].double(), sin[:T, None].double()

    def rot(t):
        a, b = t.chunk(2, -1)
        return torch.cat((a * c - b * s, a * s + b * c), -1)

    q, k, v = ((x @ w.t()).view(B, T, h, -1) for w, h in ((wq, H), (wk, KVH), (wv, KVH)))
    q, k, v = rot(q).transpose(1, 2), rot(k).transpose(1, 2), v.transpose(1, 2)
    k, v = (t.repeat_interleave(H // KVH, 1) for t in (k, v))
    future = torch.ones(T, T, dtype=torch.bool, device=x.device).triu(1)
    p = ((q @ k.transpose(2, 3)) / q.shape[-1] ** 0.5).masked_fill(future, -float("inf")).softmax(-1)
    return (p @ v).transpose(1, 2).reshape(B, T, -1) @ wo.t()


# The 16-bit roundings on the longest path to an output or gradient: each moves its tensor by at most u in the 2-norm
# (u = 2^-8 in bf16, 2^-11 in fp16), the products that follow carry that on as they carry the tensor, and independent
# roundings add up in squares, so n of them give at most sqrt(n) u.
def _assert_close_to_float64(names, got, modules, exact, n, dtype):
    u = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    for name, a, b, ref in zip(names, got, modules, exact):
        mine, theirs = _rel(a, ref), _rel(b, ref)
        print(f"  {name}: {mine:.2e}, modules {theirs:.2e}, bound {n**0.5 * u:.2e}", flush=True)
        assert mine <= n**0.5 * u, name
        assert mine <= 1.1 * theirs, name  # no term may be worse than in the modules, which round more


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B, T, H, KVH, hd", [(2, 200, 12, 4, 64), (3, 65, 2, 2, 64), (1, 1030, 8, 2, 32)])
def test_attention_layer_matches_float64(B, T, H, KVH, hd, dtype):
    print(f"\n[case] attention layer against float64 B={B} T={T} H={H} KVH={KVH} hd={hd} {dtype}", flush=True)
    m, (cos, sin) = _attention(H, KVH, hd, T, rope_kernel="hip")
    x = torch.randn(B, T, H * hd, device="cuda").to(dtype).requires_grad_()
    dy = torch.randn(B, T, H * hd, device="cuda").to(dtype)
    ins = [t.detach().double().requires_grad_() for t in (x, m.wq.weight, m.wk.weight, m.wv.weight, m.wo.weight)]
    y = _attention64(ins[0], cos, sin, H, KVH, *ins[1:])
    exact = (y.detach(), *torch.autograd.grad(y, ins, dy.double()))
    # dwq, dwk: weights, product, rotation of q and of k; P and O; the output weight, dO, dS, dq or dk, its rotation
    _assert_close_to_float64(("y", "dx", "dwq", "dwk", "dwv", "dwo"), _run(m, (x, cos, sin), dy, dtype),
                             _run(_modules_only(m), (x, cos, sin), dy, dtype), exact, 13, dtype)


def test_attention_layer_frozen_parts_and_repeated_backward():
    m, (cos, sin) = _attention(4, 2, 64, 70, rope_kernel="hip")
    x = torch.randn(2, 70, 256, device="cuda", requires_grad=True)  # fp32 in, cast by the layer
    m.wk.weight.requires_grad_(False)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = m(x, cos, sin)
    y.float().square().sum().backward(retain_graph=True)
    first = [t.grad.clone() for t in (x, m.wq.weight, m.wv.weight, m.wo.weight)]
    assert x.grad.dtype == torch.float32 and m.wk.weight.grad is None
    y.float().square().sum().backward()
    for a, t in zip(first, (x, m.wq.weight, m.wv.weight, m.wo.weight)):
        assert torch.equal(a + a, t.grad)
    for p in m.parameters():
        p.requires_grad_(False)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        (gx,) = torch.autograd.grad(m(x, cos, sin).float().square().sum(), x)
    assert torch.equal(gx, first[0])
    m.wo.weight.requires_grad_(True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        (gw,) = torch.autograd.grad(m(x.detach(), cos, sin).float().square().sum(), m.wo.weight)
    assert torch.equal(gw, first[3])


def test_attention_layer_recorded_backward():
    # the gradient of wo's gradient norm with respect to the attention's inputs, which passes through the attention's
    # first derivative only: as with the modules
    m, (cos, sin) = _attention(4, 2, 32, 33, rope_kernel="hip")
    x = torch.randn(2, 33, 128, device="cuda", requires_grad=True)
    out = []
    for mod in (m, _modules_only(m)):
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = mod(x, cos, sin)
        (gw,) = torch.autograd.grad(y.float().sum(), mod.wo.weight, create_graph=True)
        out.append(torch.autograd.grad(gw.square().sum(), x))
    for a, b in zip(*out):
        torch.testing.assert_close(a, b, rtol=5e-2, atol=5e-2 * b.abs().max().item())


def _mlp(d, ff):
    torch.manual_seed(0)
    return MLP(ModelConfig(n_layers=1, d_model=d, n_heads=1, n_kv_heads=1, d_ff=ff, attn_kernel="hip_bthd")).cuda()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape, d, ff", [((2, 200), 96, 264), ((1, 1), 64, 8), ((700,), 768, 2048), ((3, 5, 7), 40, 72)])
def test_mlp_layer_matches_its_modules(shape, d, ff, dtype):
    from nanonemo_amd.kernels.hip import layers

    print(f"\n[case] MLP layer {shape} d={d} ff={ff} {dtype}", flush=True)
    m = _mlp(d, ff)
    x = torch.randn(*shape, d, device="cuda").to(dtype).requires_grad_()
    dy = torch.randn(*shape, d, device="cuda").to(dtype)
    ref_m = _modules_only(m)
    with torch.autocast("cuda", dtype=dtype):
        assert layers.can_fuse_mlp(x, m.w_gate, m.w_up, m.w_down)
        assert not layers.can_fuse_mlp(x, ref_m.w_gate, ref_m.w_up, ref_m.w_down)
    got, ref = _run(m, (x,), dy, dtype), _run(ref_m, (x,), dy, dtype)
    # the same 16-bit products with other sums; the reference rounds silu(g), each gradient product and dW too
    tol = 2e-2 if dtype == torch.bfloat16 else 3e-3
    for name, a, b in zip(("y", "dx", "dw_gate", "dw_up", "dw_down"), got, ref):
        assert a.shape == b.shape and a.dtype == b.dtype, name
        torch.testing.assert_close(a, b, rtol=tol, atol=tol * b.abs().max().item(), msg=name)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows, d, ff", [(400, 96, 264), (700, 768, 2048), (105, 40, 72)])
def test_mlp_layer_matches_float64(rows, d, ff, dtype):
    print(f"\n[case] MLP layer against float64 {rows} d={d} ff={ff} {dtype}", flush=True)
    m = _mlp(d, ff)
    x = torch.randn(rows, d, device="cuda").to(dtype).requires_grad_()
    dy = torch.randn(rows, d, device="cuda").to(dtype)
    ins = [t.detach().double().requires_grad_() for t in (x, m.w_gate.weight, m.w_up.weight, m.w_down.weight)]
    y = (torch.nn.functional.silu(ins[0] @ ins[1].t()) * (ins[0] @ ins[2].t())) @ ins[3].t()
    exact = (y.detach(), *torch.autograd.grad(y, ins, dy.double()))
    # dx: the gate's and up's weights and products, the down weight, dh, dgate and dup, dx
    _assert_close_to_float64(("y", "dx", "dw_gate", "dw_up", "dw_down"), _run(m, (x,), dy, dtype), _run(_modules_only(m), (x,), dy, dtype),
                             exact, 9, dtype)


@pytest.mark.parametrize("kw", [dict(attn_kernel="hip_bthd", rope_kernel="hip", norm_kernel="hip"), dict(attn_kernel="hip")])
def test_model_under_inference_mode(kw):
    from nanonemo_amd.model import NanoNemo

    torch.manual_seed(0)
    m = NanoNemo(ModelConfig(n_layers=2, d_model=256, n_heads=4, n_kv_heads=2, d_ff=512, vocab_size=512, max_seq_len=96, **kw)).cuda()
    idx = torch.randint(0, 512, (2, 96), device="cuda")
    out = []
    for mode in (torch.no_grad, torch.inference_mode):
        with mode(), torch.autocast("cuda", dtype=torch.bfloat16):
            out.append(m(idx, torch.roll(idx, -1, 1)))
    assert all(torch.equal(a, b) for a, b in zip(*out))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T, F", [(1, 8), (3, 104), (129, 2048)])
def test_swiglu_matches_float64(T, F, dtype):
    from nanonemo_amd.kernels.hip import lib

    code = {torch.float16: 0, torch.bfloat16: 1}[dtype]
    g = torch.Generator(device="cuda").manual_seed(T + F)
    gu = (4 * torch.randn(T, 2 * F, device="cuda", generator=g)).to(dtype)
    edge = torch.tensor([0.0, -0.0, 60.0, -60.0, -1000.0, 1000.0, float("inf"), float("nan")], device="cuda").to(dtype)
    gu[-1, :8] = edge
    dh = torch.randn(T, F, device="cuda", generator=g).to(dtype)
    h, dgu = torch.empty_like(dh), torch.empty_like(gu)
    st = torch.cuda.current_stream().cuda_stream
    assert lib().nn_swiglu_fwd(gu.data_ptr(), h.data_ptr(), T, F, code, st) == 0
    assert lib().nn_swiglu_bwd(dh.data_ptr(), gu.data_ptr(), dgu.data_ptr(), T, F, code, st) == 0
    x = gu.double().requires_grad_()
    ref = torch.nn.functional.silu(x[:, :F]) * x[:, F:]
    (rg,) = torch.autograd.grad(ref, x, dh.double())
    # one rounding to the 16-bit type (2^-9 / 2^-12 relative, subnormals below), and a few fp32 ones
    eps, tiny = (2.0**-8, 1e-37) if dtype == torch.bfloat16 else (2.0**-11, 2.0**-24)
    big = torch.finfo(dtype).max
    for a, b in ((h, ref.detach()), (dgu, rg)):
        ok = b.isfinite() & (b.abs() < big)
        # silu'(g) cancels near its zero at g = -1.28: its fp32 error is a few 2^-24 of 1
        assert ((a.double() - b)[ok].abs() <= eps * b[ok].abs() + tiny + 1e-6).all()
        assert torch.equal(a.isnan(), b.isnan())


def _saved_through(unpack, f):
    """The gradients of f() = (output, inputs) with every saved tensor passed through unpack."""
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        y, ins = f()
    return torch.autograd.grad(y.float().square().sum(), ins)


@pytest.mark.parametrize("what", ["attention layer", "mlp", "head", "projection", "flash_attn", "flash_attn_bthd", "flash_attn_bthd_rope"])
def test_saved_tensors_are_checked_like_inputs(what):
    # what a saved-tensor hook hands back reaches the kernels by address: dense or not it is read rightly, and a host tensor
    # or another type is an error before any launch
    from nanonemo_amd.kernels.hip import flash_attn as fa
    from nanonemo_amd.kernels.hip import head, layers, linear

    torch.manual_seed(1)
    m, (cos, sin) = _attention(4, 2, 64, 70, rope_kernel="hip")
    mlp, x = _mlp(256, 264), torch.randn(2, 70, 256, device="cuda").bfloat16().requires_grad_()
    targets = torch.randint(0, 264, (2, 70), device="cuda")
    q, k, v = (torch.randn(2, 70, h, 64, device="cuda").bfloat16().requires_grad_() for h in (4, 2, 2))

    def f():
        with torch.autocast("cuda", dtype=torch.bfloat16):
            if what == "attention layer":
                return layers.attention_layer(x, cos, sin, 4, 2, m.wq, m.wk, m.wv, m.wo), (x, *m.parameters())
            if what == "mlp":
                return layers.mlp_layer(x, mlp.w_gate, mlp.w_up, mlp.w_down), (x, *mlp.parameters())
            if what == "head":
                return head.head_loss(x, mlp.w_gate, targets)[1], (x, mlp.w_gate.weight)
            if what == "projection":
                return linear.projections(x, mlp.w_gate)[0], (x, mlp.w_gate.weight)
        if what == "flash_attn":
            return fa.flash_attn(*(t.transpose(1, 2) for t in (q, k, v))), (q, k, v)
        return (fa.flash_attn_bthd(q, k, v) if what == "flash_attn_bthd" else fa.flash_attn_bthd_rope(q, k, v, cos, sin)), (q, k, v)

    def spread(t):  # the same values, every second element of a buffer
        return t if t.dim() == 0 else torch.stack((t, t), -1)[..., 0]

    ref = _saved_through(lambda t: t, f)
    for a, b in zip(_saved_through(spread, f), ref):
        # (the library may take another product for other strides: two bf16 roundings apart)
        assert torch.equal(a, b) or not what.startswith("flash") and _rel(a, b.double()) < 2 * 2.0**-8
    for bad in (lambda t: t.cpu(), lambda t: t.float() if t.dtype == torch.bfloat16 else t):
        with pytest.raises(RuntimeError):
            _saved_through(bad, f)
