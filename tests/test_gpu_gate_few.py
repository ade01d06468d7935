"""The gate gradient of up to 64 tokens, at the edges of its tiling: 16-row
blocks that end early, columns past D, whole groups past D, one and two k-steps
and the first token count past them, code-book formats.

Bound, against fp64: dW is an fp32 sum of m products, a thread's dot 16 more
steps and the sums over a workgroup at most 8 + the row blocks of its split, all
relative to the magnitudes summed; a candidate's dot sums its codes apart
from their offset, up to four times the run's largest weight."""

import pytest
import torch

from oracle import blocks, cdequant

pytestmark = pytest.mark.gpu

GGML = {"Q8_0": 8, "Q2_K": 10, "Q3_K": 11, "Q4_K": 12, "Q5_K": 13, "Q6_K": 14, "IQ3_S": 21, "IQ2_XXS": 16}
SIX = ["Q2_K", "Q3_K", "Q4_K", "Q5_K", "Q6_K", "Q8_0"]


@pytest.mark.parametrize("m,n,d,d_pad,types", [
    (1, 8, 8, 256, ["Q3_K"]),
    (31, 24, 264, 1024, SIX),
    (32, 272, 776, 776 + 248, SIX),
    (33, 40, 1288, 1536, ["Q6_K", "IQ3_S", "IQ2_XXS"]),
    (64, 1032, 2048, 2048, SIX),
    (61, 16, 4352, 4352, ["Q8_0"] * 16),
    (65, 40, 1288, 1536, SIX),
])
@pytest.mark.parametrize("with_dx", [True, False])
def test_gate_gradient_of_few_tokens(m, n, d, d_pad, types, with_dx):
    from voodoo_quant import _hip

    g = torch.Generator().manual_seed(m + n)
    qbs = []
    for qt in types:
        nb = n * d_pad // 256 * (8 if qt == "Q8_0" else 1)
        q = torch.randint(0, 256, (nb, blocks.BLOCK_BYTES[qt]), dtype=torch.uint8, generator=g)
        for off in blocks.F16_OFFSETS[qt]:
            q[:, off + 1] = (q[:, off + 1] & 0x83) | 0x28
        qbs.append(q)
    cands = [torch.from_numpy(cdequant.oracle_dequant(t, q.numpy(), n * d_pad).reshape(n, d_pad)).double()
             for t, q in zip(types, qbs)]
    x = torch.randn(m, d, generator=g).to(torch.bfloat16)
    dy = torch.randn(m, n, generator=g).to(torch.bfloat16)
    ids = [GGML[t] for t in types]
    qd = [q.reshape(-1).cuda() for q in qbs]
    probs = torch.softmax(torch.randn(len(types), generator=g), 0).cuda()
    w = _hip.mix_weight(ids, qd, probs, n, d_pad) if with_dx else None
    dx = torch.empty(m, d, dtype=torch.bfloat16, device="cuda") if with_dx else None
    ws = torch.empty(_hip.bwd_workspace_bytes(m, n, d, d_pad, len(types), False), dtype=torch.uint8, device="cuda")
    runs = []
    for _ in range(2):
        ws.fill_(255)  # nothing is read that the call did not write
        dp = torch.full((len(types),), float("nan"), device="cuda")
        _hip.gated_linear_bwd(dy.cuda(), x.cuda(), ids, qd, probs, n, d_pad, w, dx, dp, ws)
        runs.append(dp.cpu())
    assert torch.equal(runs[0], runs[1])
    dw = dy.double().t() @ x.double()
    mags = dy.double().abs().t() @ x.double().abs()
    for k, c in enumerate(cands):
        top = c.abs().view(n, -1, 16).amax(-1, keepdim=True).expand(-1, -1, 16).reshape(n, d_pad)[:, :d]
        err = (runs[0][k].double() - (dw * c[:, :d]).sum()).abs()
        assert err <= (m + 64) * 2.0**-24 * 4 * (mags * top).sum(), (k, types[k])
    if with_dx:
        want = dy.double() @ w.double().cpu()[:, :d]
        assert (dx.double().cpu() - want).norm() <= 2.0**-8 * want.norm() + 1e-12


def test_gate_gradient_ignores_padding():
    """Infinite and NaN weights in whole runs past D do not reach the gradient."""
    from voodoo_quant import _hip

    m, n, d, d_pad = 5, 24, 288, 512
    g = torch.Generator().manual_seed(2)
    q = torch.randint(0, 256, (n, d_pad // 32, 34), dtype=torch.uint8, generator=g)
    q[..., 1] = 0x28
    clean = q.clone()
    q[:, 9:12, 0], q[:, 9:12, 1] = 0, 0x7C
    q[:, 12:, 0], q[:, 12:, 1] = 1, 0x7E
    x, dy = (torch.randn(m, c, generator=g).to(torch.bfloat16).cuda() for c in (d, n))
    out = []
    for qq in (q, clean):
        ws = torch.empty(_hip.bwd_workspace_bytes(m, n, d, d_pad, 1, False), dtype=torch.uint8, device="cuda")
        dp = torch.empty(1, device="cuda")
        _hip.gated_linear_bwd(dy, x, [8], [qq.reshape(-1).cuda()], None, n, d_pad, None, None, dp, ws)
        out.append(dp.cpu())
    assert torch.equal(out[0], out[1]) and torch.isfinite(out[0]).all()


def test_group_of_one_member():
    """A stack of one member takes the tiles, whatever the token count, and gives the same gradient."""
    from voodoo_quant import _hip

    m, n, d = 7, 256, 512
    g = torch.Generator().manual_seed(9)
    q = torch.randint(0, 256, (n * d // 32, 34), dtype=torch.uint8, generator=g)
    q[:, 1] = 0x28
    qd = q.reshape(-1).cuda()
    x, dy = (torch.randn(m, c, generator=g).to(torch.bfloat16).cuda() for c in (d, n))
    one = torch.empty(1, device="cuda")
    ws = torch.empty(_hip.bwd_workspace_bytes(m, n, d, d, 1, False), dtype=torch.uint8, device="cuda")
    _hip.gated_linear_bwd(dy, x, [8], [qd], None, n, d, None, None, one, ws)
    members = [((8,), [qd], n)]
    stacked = torch.empty(1, device="cuda")
    ws = torch.empty(_hip.group_bwd_workspace_bytes(m, d, members), dtype=torch.uint8, device="cuda")
    _hip.gated_linear_group_bwd(dy, x, members, d, None, None, [stacked], ws)
    w = torch.from_numpy(cdequant.oracle_dequant("Q8_0", q.numpy(), n * d).reshape(n, d)).double()
    dw = dy.double().cpu().t() @ x.double().cpu()
    mags = dy.double().abs().cpu().t() @ x.double().abs().cpu()
    scale = (mags * w.abs().max()).sum()
    for got in (one, stacked):
        assert (got.double().cpu() - (dw * w).sum()).abs() <= (m + 64) * 2.0**-24 * 4 * scale
