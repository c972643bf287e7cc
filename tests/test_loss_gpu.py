"""GPU tests of the cross-entropy kernels and of the output layer and loss as one call (kernels/hip/head.py)."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F
from torch import nn

pytestmark = pytest.mark.gpu

DTYPES = [torch.bfloat16, torch.float16, torch.float32]


def _call(logits, targets, grad=1.0):
    from nanonemo_amd.kernels.hip import check_loss, lib

    (R, V), code = logits.shape, {torch.float16: 0, torch.bfloat16: 1, torch.float32: 2}[logits.dtype]
    lse, rows, loss, inv = (torch.empty(n, device="cuda") for n in (R, R, (), ()))
    g, d, st = torch.tensor(grad, device="cuda"), torch.empty_like(logits), torch.cuda.current_stream().cuda_stream
    L = lib()
    check_loss(L.nn_cross_entropy_fwd(logits.data_ptr(), targets.data_ptr(), lse.data_ptr(), rows.data_ptr(), loss.data_ptr(), inv.data_ptr(), R, V, code, st))
    check_loss(L.nn_cross_entropy_bwd(logits.data_ptr(), targets.data_ptr(), lse.data_ptr(), inv.data_ptr(), g.data_ptr(), d.data_ptr(), R, V, code, st))
    return lse, loss, d


# Vocabularies around the 16-byte vectors and a block's 256 threads, odd ones whose rows start anywhere, and the model's.
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("R, V", [(1, 1), (3, 7), (5, 8), (4, 63), (7, 1003), (2, 2048), (3, 2057), (33, 50304)])
def test_cross_entropy_matches_float64(R, V, dtype):
    print(f"\n[case] cross entropy R={R} V={V} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(R + V)
    logits = (3 * torch.randn(R, V, device="cuda", generator=g)).to(dtype)
    targets = torch.randint(0, V, (R,), device="cuda", generator=g)
    if R > 2:
        targets[1] = -100
        logits[0, : max(1, V // 2)] += 80  # a row dominated by large values
        if V > 1:
            logits[2, 0] = -float("inf")
            targets[2] = V - 1
    lse, loss, d = _call(logits, targets, 0.7)
    x = logits.double().requires_grad_()
    ref = F.cross_entropy(x, targets)
    (rg,) = torch.autograd.grad(ref, x, torch.tensor(0.7, device="cuda", dtype=torch.float64))
    # exp's argument is rounded twice (2^-23 of at most ~100) and log's result once
    assert (lse.double() - x.logsumexp(1)).abs().max() <= 4e-6 * max(1.0, x.detach()[x.isfinite()].abs().max().item())
    assert abs(loss.double() - ref) <= 2e-5 * max(1.0, ref.abs().item())
    # one rounding to the logits' type (fp16 has subnormals below 2^-24), and exp's argument as above
    eps, tiny = {torch.bfloat16: (2.0**-8, 1e-12), torch.float16: (2.0**-11, 2.0**-24), torch.float32: (3e-5, 1e-9)}[dtype]
    assert ((d.double() - rg).abs() <= (eps + 3e-5) * rg.abs() + tiny + 1e-7 / R).all()


@pytest.mark.parametrize("dtype", DTYPES)
def test_cross_entropy_special_values_follow_torch(dtype):
    base = torch.randn(4, 300, device="cuda").to(dtype)
    inf = float("inf")
    for what, row, targets in (("all -inf", torch.full((300,), -inf), [0, 1, 2, 3]), ("a +inf", torch.cat([torch.tensor([inf]), torch.zeros(299)]), [0, 5, 2, 3]),
                               ("a NaN", torch.cat([torch.zeros(299), torch.tensor([float("nan")])]), [0, 1, 2, 3]),
                               ("target -inf", torch.cat([torch.zeros(5), torch.full((295,), -inf)]), [0, 7, 2, 3]),
                               ("none counts", torch.zeros(300), [-100] * 4)):
        logits, t = base.clone(), torch.tensor(targets, device="cuda")
        logits[1] = row.to(dtype)
        _, loss, d = _call(logits, t)
        x = logits.float().requires_grad_()
        ref = F.cross_entropy(x, t)
        (rg,) = torch.autograd.grad(ref, x)
        assert torch.equal(loss.isnan(), ref.isnan()) and (ref.isnan() or torch.allclose(loss, ref.detach(), rtol=1e-5)), what
        assert torch.equal(d.isnan(), rg.isnan()), what
    t = torch.tensor([0, 300, 2, 3], device="cuda")  # out of range: no read past the row, and a loss that shows it
    assert _call(base, t)[1].isnan()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
def test_special_values_in_a_row_that_does_not_count_follow_torch(value, dtype):
    logits = torch.randn(3, 300, device="cuda").to(dtype)
    logits[1, 7] = value
    t = torch.tensor([0, -100, 2], device="cuda")
    _, loss, d = _call(logits, t)
    x = logits.float().requires_grad_()
    ref = F.cross_entropy(x, t)
    (rg,) = torch.autograd.grad(ref, x)
    assert torch.allclose(loss, ref.detach(), rtol=1e-5)
    assert torch.equal(d.isnan(), rg.isnan()) and (d[1].isnan() | (d[1] == 0)).all()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("bad", [-1, 300, 1 << 40])
def test_a_target_out_of_range_shows_in_the_loss_and_in_its_rows_gradient(dtype, bad):
    logits = torch.randn(4, 300, device="cuda").to(dtype)
    t = torch.tensor([0, bad, -100, 3], device="cuda")
    _, loss, d = _call(logits, t)
    assert loss.isnan() and d[1].isnan().all() and d[[0, 2, 3]].isfinite().all()


@pytest.mark.parametrize("V", [512, 1003])
def test_head_loss_matches_its_modules(V):
    from nanonemo_amd.kernels.hip import head

    torch.manual_seed(0)
    m = nn.Linear(96, V, bias=False).cuda()
    x = torch.randn(2, 70, 96, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    t = torch.randint(0, V, (2, 70), device="cuda")
    t[0, 3] = -100
    extra = 1e-4 * torch.randn(2, 70, V, device="cuda", dtype=torch.bfloat16)

    def modules():
        logits = m(x)
        return logits, F.cross_entropy(logits.float().view(-1, V), t.reshape(-1))

    out = []
    for f in (lambda: head.head_loss(x, m, t), modules):
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert head.can_fuse_head(x, m, t) and not head.can_fuse_head(x, m, t.int()) and not head.can_fuse_head(x, m, t[:1])
            logits, loss = f()
        res = [logits.detach().clone(), loss.detach(), *torch.autograd.grad(loss, (x, m.weight), retain_graph=True)]
        res += torch.autograd.grad((logits, loss), (x, m.weight), (extra, torch.tensor(0.5, device="cuda")), retain_graph=True)
        res += torch.autograd.grad(logits, (x, m.weight), extra, retain_graph=True)
        with torch.no_grad():
            logits.mul_(2.0)  # the caller's logits may change before the loss's backward
        res += torch.autograd.grad(loss, (x, m.weight))
        out.append(res)
    for i, (a, b) in enumerate(zip(*out)):
        assert a.shape == b.shape and a.dtype == b.dtype, i
        torch.testing.assert_close(a, b, rtol=2e-2, atol=2e-2 * b.abs().max().item(), msg=str(i))
    assert torch.equal(out[0][2], out[0][-2]) and torch.equal(out[0][3], out[0][-1])


def test_head_loss_frees_the_logits_with_the_backward():
    from nanonemo_amd.kernels.hip import head

    m = nn.Linear(64, 4096, bias=False).cuda()
    x, t = torch.randn(2048, 64, device="cuda"), torch.randint(0, 4096, (2048,), device="cuda")
    m.weight.grad = torch.zeros_like(m.weight)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        loss = head.head_loss(x, m, t)[1]
    held = torch.cuda.memory_allocated()
    loss.backward()
    assert held - torch.cuda.memory_allocated() >= 2048 * 4096 * 2  # with loss still referenced


def test_head_loss_second_derivative():
    from nanonemo_amd.kernels.hip import head

    torch.manual_seed(0)
    m = nn.Linear(32, 64, bias=False).cuda()
    x = torch.randn(40, 32, device="cuda", requires_grad=True)
    t = torch.randint(0, 64, (40,), device="cuda")
    out = []
    for f in (lambda: head.head_loss(x, m, t)[1], lambda: F.cross_entropy(m(x).float(), t)):
        with torch.autocast("cuda", dtype=torch.bfloat16):
            loss = f()
        (gx,) = torch.autograd.grad(loss, x, create_graph=True)
        out.append(torch.autograd.grad(gx.square().sum(), (x, m.weight)))
    for a, b in zip(*out):
        torch.testing.assert_close(a, b, rtol=3e-2, atol=3e-2 * b.abs().max().item())
