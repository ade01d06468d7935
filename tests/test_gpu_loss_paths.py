"""The distillation loss's instantiations: e^s as the square of e^(s/2) at T = 2
(threads without logits, masked logits), rows few enough for the larger
workgroup, and logits large enough to be streamed past the caches.  Against
fp64."""

import math

import pytest
import torch

from voodoo_quant import _hip

pytestmark = pytest.mark.gpu


def _ref(s, t, y, temp):
    s, t = s.double(), t.double()
    lp, lq, lt = s.log_softmax(-1), (s / temp).log_softmax(-1), (t / temp).log_softmax(-1)
    live = y != -100
    ce = -lp.gather(1, y.clamp_min(0).view(-1, 1)).view(-1)[live].mean()
    p = lt.exp()
    kl = (torch.where(p > 0, p * (lt - lq), 0.0).sum(-1) * temp * temp).mean()
    hot = torch.zeros_like(s).scatter_(1, y.clamp_min(0).view(-1, 1), 1.0)
    grad = (lp.exp() - hot) * live.view(-1, 1) / live.sum() + (lq.exp() - p) * temp / s.shape[0]
    return ce, kl, grad


@pytest.mark.parametrize("temp", [1.0, 2.0, 1.5])
@pytest.mark.parametrize("rows,vocab", [
    (5, 8),          # one thread has logits
    (7, 2056),       # one past a 256-thread pass
    (3, 65536),      # the larger workgroup, whole passes
    (6, 73736),      # the larger workgroup, a ragged last pass
    (600, 65544),    # few-row limit passed
    (1024, 65536),   # streamed
])
def test_loss_paths(rows, vocab, temp):
    g = torch.Generator(device="cuda").manual_seed(rows + vocab)
    s = (3 * torch.randn(rows, vocab, device="cuda", generator=g)).bfloat16()
    t = (s.float() + torch.randn(rows, vocab, device="cuda", generator=g)).bfloat16()
    if vocab > 8:  # masked logits: no probability on either side
        s[:, 3:7] = -math.inf
        t[:, 3:7] = -math.inf
        s[0, 8:2056] = -math.inf  # a wave whose threads see nothing else in their first pass
        t[0, 8:2056] = -math.inf
    y = torch.randint(0, 3, (rows,), device="cuda", generator=g)
    y[1] = -100
    out, ws = _hip.distill_loss_fwd(s, t, y, temp)
    grad = _hip.distill_loss_bwd(s, t, y, temp, torch.ones(2, device="cuda"), ws)
    ref_ce, ref_kl, ref = _ref(s, t, y, temp)
    # fp32 sums of up to 65536 terms of one sign (CE) or nearly so (KL)
    assert abs(float(out[0]) - float(ref_ce)) <= 1e-5 * float(ref_ce)
    assert abs(float(out[1]) - float(ref_kl)) <= 1e-5 * float(ref_kl)
    # one bf16 rounding (2^-9 of a value at most), over fp32 exponentials
    assert float((grad.double() - ref).norm() / ref.norm()) <= 4e-3
