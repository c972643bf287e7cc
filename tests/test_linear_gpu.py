"""GPU tests of the linear layers' weight gradients (nn_linear_wgrad) and of the autograd path that uses them."""

from __future__ import annotations

import ctypes

import pytest
import torch
from torch import nn

pytestmark = pytest.mark.gpu

# T: no rows, one, around a 64-token stage and a group of four, odd; N and K around the 128-wide tile and not multiples
# of it; several splits (few tiles, many tokens) and none.
WGRAD = [(0, 128, 128), (1, 8, 8), (63, 128, 64), (64, 120, 136), (65, 8, 264), (255, 256, 128), (257, 136, 120), (1000, 1280, 768),
         (5000, 264, 72), (8192, 768, 768)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T, N, K", WGRAD)
def test_wgrad_matches_float64(T, N, K, dtype):
    from nanonemo_amd.kernels.hip.linear import wgrad

    print(f"\n[case] wgrad T={T} N={N} K={K} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T + N + K)
    # wider rows than the operands, the rest NaN: columns past the width must not reach the result
    buf = [torch.full((T, n + 16), float("nan"), device="cuda", dtype=dtype) for n in (N, K)]
    dy, x = (b[:, 8 : 8 + n].copy_(torch.randn(T, n, device="cuda", generator=g)) for b, n in zip(buf, (N, K)))
    rows = [N] if N < 24 else [N - 16, 8, 8]
    got = wgrad(dy, x, rows)
    assert [tuple(t.shape) for t in got] == [(r, K) for r in rows] and all(t.dtype == torch.float32 for t in got)
    got, again = torch.cat(got), torch.cat(wgrad(dy, x, rows))
    ref = dy.double().t().contiguous() @ x.double()
    assert torch.equal(got, again)
    # products of 16-bit values are exact in fp32; T sums, each rounded once: |error| <= T 2^-24 sum |dy x|
    bound = T * 2.0**-24 * (dy.double().abs().t().contiguous() @ x.double().abs())
    assert ((got.double() - ref).abs() <= bound).all()


def test_wgrad_of_an_odd_number_of_columns_copies_nothing():
    # the output layer's gradient for a vocabulary that is no multiple of 8: 0.8 GB at 8192 x 50257
    from nanonemo_amd.kernels.hip.linear import wgrad

    T, N, K = 2048, 4099, 64
    dy, x = (torch.randn(T, n, device="cuda").bfloat16() for n in (N, K))
    wgrad(dy, x, [N])  # the library's own workspace
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    (got,) = wgrad(dy, x, [N])
    assert torch.cuda.max_memory_allocated() - before < dy.nbytes
    # any other layout is read as well: column slices, columns in memory order, a start off the 16-byte grid
    wide = torch.full((T, N + 7), float("nan"), device="cuda").bfloat16()
    off = torch.empty(T * N + 1, device="cuda", dtype=torch.bfloat16)[1:].view(T, N)
    for like in (wide[:, 3 : 3 + N], torch.empty(N, T, device="cuda", dtype=torch.bfloat16).t(), off):
        assert torch.equal(wgrad(like.copy_(dy), x, [N])[0], got)


def test_wgrad_rejects_bad_arguments_before_any_launch():
    from nanonemo_amd.kernels.hip import lib

    L = lib()
    t = torch.zeros(64, 64, device="cuda", dtype=torch.bfloat16)
    out = torch.zeros(64, 64, device="cuda")

    def call(N=64, ldy=64, rows=(64,), p=t.data_ptr(), dt=1):
        o = (ctypes.c_void_p * len(rows))(*([out.data_ptr()] * len(rows)))
        rc = L.nn_linear_wgrad(p, ldy, t.data_ptr(), 64, 64, N, 64, len(rows), o, (ctypes.c_int64 * len(rows))(*rows), None, 0, dt, None)
        return rc, L.nn_linear_last_error().decode()

    for kw, msg in ((dict(N=60, rows=(60,)), "multiples of 8"), (dict(ldy=56), "row strides"), (dict(rows=(32,)), "add up to N"),
                    (dict(p=t.data_ptr() + 2), "16-byte aligned"), (dict(dt=2), "float16 or bfloat16"), (dict(rows=(16,) * 4), "1 to 3 outputs")):
        rc, err = call(**kw)
        assert rc != 0 and msg in err, (kw, err)


def _layers(K, ns):
    torch.manual_seed(0)
    return [nn.Linear(K, n, bias=False).cuda() for n in ns]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("xdt", [torch.float32, None])
def test_projections_match_autocast_linears(dtype, xdt):
    from nanonemo_amd.kernels.hip import linear

    layers = _layers(96, (64, 32, 8))
    x = torch.randn(3, 50, 96, device="cuda", dtype=xdt or dtype, requires_grad=True)
    dys = [torch.randn(3, 50, n, device="cuda", dtype=dtype) for n in (64, 32, 8)]
    with torch.autocast("cuda", dtype=dtype):
        assert linear.can_project(x, *layers)
        got, ref = linear.projections(x, *layers), [m(x) for m in layers]
    ins = (x, *(m.weight for m in layers))
    gg, gr = torch.autograd.grad(got, ins, dys), torch.autograd.grad(ref, ins, dys)
    # the same 16-bit products, other sums; the reference also rounds each gradient to 16 bits
    tol = 2e-2 if dtype == torch.bfloat16 else 3e-3
    for a, b in zip((*got, *gg), (*ref, *gr)):
        assert a.shape == b.shape and a.dtype == b.dtype
        torch.testing.assert_close(a, b, rtol=tol, atol=tol * b.abs().max().item())
    # an unused output and a frozen weight
    layers[1].weight.requires_grad_(False)
    with torch.autocast("cuda", dtype=dtype):
        a, _, c = linear.projections(x, *layers)
    (a.float().sum() + c.float().sum()).backward()
    assert layers[1].weight.grad is None and layers[0].weight.grad.dtype == torch.float32 and x.grad.dtype == x.dtype


def test_projections_second_derivative():
    from nanonemo_amd.kernels.hip import linear

    (m,) = _layers(32, (16,))
    x = torch.randn(40, 32, device="cuda", requires_grad=True)
    out = []
    for f in (lambda: linear.projections(x, m)[0], lambda: m(x)):
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = f()
        (gx,) = torch.autograd.grad(y.float().square().sum(), x, create_graph=True)
        out.append(torch.autograd.grad(gx.square().sum(), (x, m.weight)))
    for a, b in zip(*out):
        torch.testing.assert_close(a, b, rtol=3e-2, atol=3e-2 * b.abs().max().item())


def test_only_untouched_layers_under_autocast_take_the_path():
    from nanonemo_amd.kernels.hip import linear

    (m,) = _layers(32, (16,))
    x = torch.randn(4, 32, device="cuda")
    assert not linear.can_project(x, m)  # no autocast
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert linear.can_project(x, m)
        assert not linear.can_project(x.cpu(), m) and not linear.can_project(x.double(), m) and not linear.can_project(x[:0], m)
        assert not linear.can_project(torch.nested.nested_tensor([x, x]), m)
        h = m.register_forward_hook(lambda *_: None)
        assert not linear.can_project(x, m)
        h.remove()
        assert linear.can_project(x, m)
        assert not linear.can_project(x, nn.Linear(32, 16).cuda()) and not linear.can_project(x, nn.Linear(32, 12, bias=False).cuda())
        nn.utils.parametrizations.weight_norm(m)
        assert not linear.can_project(x, m)
        with torch.autograd.forward_ad.dual_level():
            assert not linear.can_project(x, _layers(32, (16,))[0])
        assert not linear.can_project(x, nn.Linear(32, 16, bias=False).cuda().bfloat16())


@pytest.mark.parametrize("what", ["offset", "row stride", "column stride"])
def test_wgrad_copies_what_the_kernel_cannot_read(what):
    from nanonemo_amd.kernels.hip.linear import wgrad

    T, N, K = 130, 64, 40
    t = torch.randn(2 * T * (N + 4) + 3, device="cuda").bfloat16()
    dy = {"offset": t[3 : 3 + T * N].view(T, N), "row stride": t[: T * (N + 4)].view(T, N + 4)[:, :N],
          "column stride": t[: T * N].view(N, T).t()}[what]
    x = torch.randn(T, K, device="cuda").bfloat16()
    assert torch.equal(wgrad(dy, x, [N])[0], wgrad(dy.clone(memory_format=torch.contiguous_format), x, [N])[0])
    (got,), (ref,) = wgrad(x, dy, [K]), wgrad(x, dy.clone(memory_format=torch.contiguous_format), [K])
    assert torch.equal(got, ref)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shapes", [[(8, 8)], [(72, 56), (8, 200), (136, 64)], [(1280, 768), (64, 64), (128, 8), (16, 328)]])
def test_cast_both_is_exact(shapes, dtype):
    from nanonemo_amd.kernels import hip

    ws = [torch.randn(s, device="cuda") for s in shapes]
    dst = [torch.full(s, float("nan"), device="cuda", dtype=dtype) for s in shapes]
    ldt = [r + 8 * (i % 2) for i, (r, _) in enumerate(shapes)]
    turned = [torch.full((c, ld), float("nan"), device="cuda", dtype=dtype) for (_, c), ld in zip(shapes, ldt)]
    n = len(ws)
    ptrs = [(ctypes.c_void_p * n)(*(t.data_ptr() for t in ts)) for ts in (ws, dst, turned)]
    sizes = [(ctypes.c_int64 * n)(*v) for v in ([r for r, _ in shapes], [c for _, c in shapes], ldt)]
    stream = torch.cuda.current_stream().cuda_stream
    code = hip.DTYPE_BF16 if dtype is torch.bfloat16 else hip.DTYPE_F16
    assert hip.lib().nn_linear_cast_both(n, *ptrs, *sizes, code, stream) == 0
    for w, d, t, (r, _) in zip(ws, dst, turned, shapes):
        assert torch.equal(d, w.to(dtype))
        assert torch.equal(t[:, :r], w.to(dtype).t())
        assert t[:, r:].isnan().all()
    sizes[0][0] = 4  # not a multiple of 8
    assert hip.lib().nn_linear_cast_both(n, *ptrs, *sizes, code, stream) != 0
