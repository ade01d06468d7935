"""Edges of the 256x256 products' stream: reductions shorter than its three
stages and ending inside one, ragged rows and columns, tiles split along K,
several tiles per workgroup (forward), and single-token to odd-token gate
products.  Against fp64 products of the same bf16 operands."""

import pytest
import torch

from oracle import mixture
from voodoo_quant import _hip, rtn

pytestmark = pytest.mark.gpu

# One bf16 rounding of each output: at most 2^-9 of a value, 2^-9 / sqrt(3) = 1.1e-3 of the norm when the roundings
# are uniform; the fp32 sums add under 1e-6 (K <= 2048 terms).  2e-3 also covers the fixed-order fp32 parts.
REL = 2e-3


@pytest.mark.parametrize("split", [True, False], ids=["split", "whole"])
@pytest.mark.parametrize("m,n,d", [
    (3073, 4104, 8),      # one chunk of k: a stage of 8, two of zeros
    (3073, 4104, 64),     # exactly one stage
    (3001, 4360, 72),     # one stage and a chunk
    (3072, 4096, 192),    # three whole stages, no ragged edge
    (3000, 8200, 200),    # two rounds of tiles, the next tile's copies behind a partial stage
    (8192, 2064, 2048),   # split tail tiles
])
def test_forward_edges(m, n, d, split):
    g = torch.Generator(device="cuda").manual_seed(m + n + d)
    x = torch.randn(m, d, device="cuda", generator=g).bfloat16()
    d_pad = (d + 255) // 256 * 256
    w = torch.full((n, d_pad), float("nan"), device="cuda", dtype=torch.bfloat16)  # columns past d are never read
    w[:, :d] = torch.randn(n, d, device="cuda", generator=g).bfloat16()
    y = torch.full((m, n), float("nan"), device="cuda", dtype=torch.bfloat16)
    nbytes = _hip.fwd_workspace_bytes(m, n, d)
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda") if split and nbytes else None
    _hip.linear_fwd(x, w, n, y, ws)
    ref = x.double() @ w[:, :d].double().t()
    assert float((y.double() - ref).norm() / ref.norm()) < REL


@pytest.mark.parametrize("m", [1, 63, 64, 65, 193, 1000])
@pytest.mark.parametrize("n,d", [(8, 8), (264, 520), (1000, 256), (256, 1032)])
def test_backward_edges(m, n, d):
    types, ids = ["Q8_0", "Q6_K", "Q5_K", "Q4_K", "Q3_K", "Q2_K"], [8, 14, 13, 12, 11, 10]
    g = torch.Generator().manual_seed(m + n + d)
    d_pad = (d + 255) // 256 * 256
    src = torch.zeros(n, d_pad)
    src[:, :d] = torch.randn(n, d, generator=g) * 0.02
    qb = [rtn.rtn_quantize_tensor(src, t).reshape(-1).cuda() for t in types]
    cands = [_hip.dequant(i, q, n, d_pad)[:, :d].cpu() for i, q in zip(ids, qb)]
    probs = torch.softmax(torch.randn(len(ids), generator=g), 0)
    x, dy = (torch.randn(m, k, generator=g).bfloat16() for k in (d, n))
    w = mixture.mix_weight(cands, probs).bfloat16()
    w_eff = torch.zeros(n, d_pad, dtype=torch.bfloat16)
    w_eff[:, :d] = w
    dx = torch.full((m, d), float("nan"), dtype=torch.bfloat16, device="cuda")
    dp = torch.empty(len(ids), device="cuda")
    ws = torch.empty(_hip.bwd_workspace_bytes(m, n, d, d_pad, len(ids), False), dtype=torch.uint8, device="cuda")
    _hip.gated_linear_bwd(dy.cuda(), x.cuda(), ids, qb, probs.cuda(), n, d_pad, w_eff.cuda(), dx, dp, ws)
    ref = dy.double() @ w.double()
    assert float((dx.cpu().double() - ref).norm() / ref.norm()) < REL
    dw = dy.double().t() @ x.double()
    ref_dp = torch.stack([(dw * c.double()).sum() for c in cands])
    # fp32 dots of at most 256 x 256 terms per partial, summed in fp64: against the terms' own size
    scale = torch.stack([(dw * c.double()).norm() for c in cands])
    assert bool(((dp.cpu().double() - ref_dp).abs() <= 1e-5 * scale + 1e-5 * ref_dp.abs()).all())
