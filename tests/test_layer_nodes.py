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
    assert not any(isinstance(v, torch.Tensor) and v.numel() >= logits.numel() for v in vars(node).values())
    with pytest.raises(RuntimeError, match="freed"):
        node.saved_tensors
