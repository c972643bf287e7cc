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
