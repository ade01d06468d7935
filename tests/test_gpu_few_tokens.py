"""The forward of up to 8 tokens in the mixture's own pass, with and without
W_eff in memory, at the edges of its work split: rows that end inside a
workgroup's 16 groups, a partial last workgroup, columns past D, and the first
token count that goes to the general path.  Every tensor is small enough for
the pass to be taken at each count up to 8.

Bounds: an output is one bf16 rounding (2^-8 of its value, at most) of an fp32
sum of D products, each rounded once and each partial sum once: 2^-24 of the
sum of the products' magnitudes per step, and there are fewer than 64 steps
from a product to the result (16 in a thread, 4 across its group, up to
D / 4096 + 4 across groups)."""

import pytest
import torch

from oracle import blocks, cdequant

pytestmark = pytest.mark.gpu

GGML = {"Q8_0": 8, "Q2_K": 10, "Q3_K": 11, "Q4_K": 12, "Q5_K": 13, "Q6_K": 14, "IQ3_S": 21}
SIX = ["Q2_K", "Q3_K", "Q4_K", "Q5_K", "Q6_K", "Q8_0"]


def _candidates(types, rows, cols, seed):
    g = torch.Generator().manual_seed(seed)
    out = []
    for qt in types:
        nb = rows * cols // 256 * (8 if qt == "Q8_0" else 1)
        q = torch.randint(0, 256, (nb, blocks.BLOCK_BYTES[qt]), dtype=torch.uint8, generator=g)
        for off in blocks.F16_OFFSETS[qt]:  # normal fp16 scales
            q[:, off + 1] = (q[:, off + 1] & 0x83) | 0x28
        out.append(q)
    return out


def _close(y, exact, mags):
    bound = exact.abs() * 2.0**-8 + 64 * 2.0**-24 * mags + 1e-30
    worst = ((y.double().cpu() - exact).abs() / bound).max().item()
    assert worst <= 1.0, worst


@pytest.mark.parametrize("m,n,d,d_pad,types", [
    (1, 8, 8, 256, ["Q4_K"]),                      # one unit, one thread's half run
    (1, 24, 776, 1024, SIX),                       # 4 groups a row; D ends inside the last one
    (2, 40, 1288, 1536, SIX),                      # 6 groups a row: rows straddle workgroups, the last is partial
    (3, 16, 4352, 4352, ["Q3_K", "Q6_K", "Q8_0"]),  # 17 groups a row
    (4, 8, 264, 1024, SIX),                        # whole groups past D
    (5, 104, 2048, 2048, ["Q5_K", "IQ3_S", "Q8_0"]),
    (8, 272, 5120, 5120, SIX),
    (8, 72, 256, 256, ["Q8_0"] * 16),              # the largest staging: 68 KiB
    (9, 24, 776, 1024, SIX),                       # general path
])
def test_few_token_forward(m, n, d, d_pad, types):
    from voodoo_quant import _hip

    qbs = _candidates(types, n, d_pad, 7 * m + n)
    ids = [GGML[t] for t in types]
    g = torch.Generator().manual_seed(m)
    probs = torch.softmax(torch.randn(len(types), generator=g), 0)
    x = torch.randn(m, d, generator=g).to(torch.bfloat16)
    cands = [torch.from_numpy(cdequant.oracle_dequant(t, q.numpy(), n * d_pad).reshape(n, d_pad)).double()
             for t, q in zip(types, qbs)]
    qd = [q.reshape(-1).cuda() for q in qbs]
    xd, pd = x.cuda(), probs.cuda()
    # W_eff kept: the mixture's bits, and the product of its bf16 values
    w = torch.full((n, d_pad), float("nan"), dtype=torch.bfloat16, device="cuda")
    y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    ws = torch.empty(max(1, _hip.fwd_workspace_bytes(m, n, d)), dtype=torch.uint8, device="cuda")
    _hip.gated_linear_fwd(xd, ids, qd, pd, n, d_pad, w, y, ws)
    mixed = _hip.mix_weight(ids, qd, pd, n, d_pad)
    assert torch.equal(w.view(torch.int16), mixed.view(torch.int16))
    wd = mixed.double().cpu()[:, :d]
    _close(y, x.double() @ wd.t(), x.double().abs() @ wd.abs().t())
    # W_eff never in memory
    if m <= 8:
        y2 = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
        wf = torch.empty(max(1, _hip.fused_workspace_bytes(m, n, d, False)), dtype=torch.uint8, device="cuda")
        _hip.gated_linear_fwd_fused(xd, ids, qd, pd, n, d_pad, y2, wf)
        pk = probs.double()
        exact = sum(p * c for p, c in zip(pk, cands))[:, :d]
        # K fma steps and their scale products come on top, relative to sum p |W| and the codes' offsets
        # (a code's offset is at most 128 of 255 units: under twice the largest |weight| of its run)
        size = sum(p * c.abs().view(n, -1, 16).amax(-1, keepdim=True).expand(-1, -1, 16).reshape(n, d_pad)
                   for p, c in zip(pk, cands))[:, :d]
        mags = x.double().abs() @ (4 * size).t()
        _close(y2, x.double() @ exact.t(), mags)


def test_few_token_forward_ignores_weights_past_d_and_zero_workspace():
    """Infinite padding weights do not reach y; without a workspace the call takes the general path."""
    from voodoo_quant import _hip

    n, d, d_pad, m = 16, 264, 512, 2
    q = _candidates(["Q8_0"], n, d_pad, 3)[0].view(n, d_pad // 32, 34)
    q[:, 9:, 0], q[:, 9:, 1] = 0, 0x7C  # inf scales of the blocks past column 288
    x = torch.randn(m, d, generator=torch.Generator().manual_seed(0)).to(torch.bfloat16).cuda()
    p = torch.ones(1, device="cuda")
    ys = []
    for ws in (torch.empty(_hip.fwd_workspace_bytes(m, n, d), dtype=torch.uint8, device="cuda"), None):
        w = torch.empty(n, d_pad, dtype=torch.bfloat16, device="cuda")
        y = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
        _hip.gated_linear_fwd(x, [8], [q.reshape(-1).cuda()], p, n, d_pad, w, y, ws)
        ys.append(y.float().cpu())
    assert torch.isfinite(ys[0]).all()
    assert (ys[0] - ys[1]).norm() <= 2.0**-7 * ys[1].norm()
