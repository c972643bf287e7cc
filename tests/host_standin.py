"""A CPU stand-in for the layers' functions of the host module (csrc/host.cpp), in plain torch, so that the autograd
nodes around them (kernels/hip/head.py, layers.py, linear.py) can be tested without a GPU."""

from __future__ import annotations

import torch
import torch.nn.functional as F

from nanonemo_amd.kernels import hip


def _reads(*ts):
    """The kernels read raw addresses: a tensor without storage of its own (a batched one) is an error."""
    for t in ts:
        if t is not None:
            t.data_ptr()


class Host:
    def __getattr__(self, name):  # whatever needs no GPU is the module's own
        return getattr(hip.host(), name)

    def wgrad(self, dy, x, rows):
        _reads(dy, x)
        return list((dy.float().t() @ x.float()).split(rows))

    def project_fwd(self, x, ws, turned):
        w = torch.cat([w.to(x.dtype) for w in ws])
        return x @ w.t(), w

    def mlp_fwd(self, x, w_gate, w_up, w_down, turned):
        w, wd = torch.cat([w_gate, w_up]).to(x.dtype), w_down.to(x.dtype)
        gu = x @ w.t()
        g, u = gu.float().chunk(2, 1)
        h = (F.silu(g) * u).to(x.dtype)
        return h @ wd.t(), gu, h, w, wd

    def mlp_bwd(self, dy, x, gu, h, w, wd, need_x, need_gu, need_down):
        _reads(dy)
        dh = (dy @ wd).float()
        g, u = gu.float().chunk(2, 1)
        s = torch.sigmoid(g)
        dgu = torch.cat([dh * u * s * (1 + g * (1 - s)), dh * g * s], 1).to(x.dtype)
        dws = self.wgrad(dgu, x, [h.shape[1]] * 2) if need_gu else [None, None]
        return [dgu @ w if need_x else None, *dws, self.wgrad(dy, h, [wd.shape[0]])[0] if need_down else None]

    def head_fwd(self, x, w, targets, turned):
        w16 = w.to(x.dtype)
        logits = x @ w16.t()
        lse = logits.float().logsumexp(1)
        return logits, F.cross_entropy(logits.float(), targets), w16, lse, 1 / (targets != -100).sum().float()

    def head_bwd(self, dlogits, dloss, logits, x, w, targets, lse, inv, need_x, need_w):
        _reads(dlogits, dloss)
        d = dlogits
        if dloss is not None:
            self.recomputed = logits is None
            logits = x @ w.t() if logits is None else logits
            counts = (targets != -100).unsqueeze(1)
            p = (logits.float() - lse.unsqueeze(1)).exp() - F.one_hot(targets.clamp_min(0), logits.shape[1])
            t = (p * counts * dloss * inv).to(x.dtype)
            d = t if d is None else t + d
        return [d @ w if need_x else None, self.wgrad(d, x, [w.shape[0]])[0] if need_w else None]


def install(monkeypatch) -> Host:
    """Make the layers' nodes call the stand-in; returns it."""
    from nanonemo_amd.kernels.hip import head, layers, linear

    h = Host()
    for m in (head, layers, linear):
        monkeypatch.setattr(m, "host", lambda: h)
    return h
