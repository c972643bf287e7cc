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
