"""Embedding rows where several requested rows share a workgroup: row widths
that leave slots over, spans whose last 16-byte chunk is the buffer's end, ids
out of range beside valid ones, and rows of more than one segment."""

import pytest
import torch

from oracle import blocks, cdequant

pytestmark = pytest.mark.gpu

GGML = {"Q8_0": 8, "Q2_K": 10, "Q3_K": 11, "Q4_K": 12, "Q5_K": 13, "Q6_K": 14, "IQ3_S": 21}


@pytest.mark.parametrize("dim,vocab,nids,types", [
    (8, 5, 33, ["Q3_K", "Q8_0"]),            # 16 rows a workgroup, half a thread's run
    (256, 3, 1, ["Q3_K"]),                   # an odd count of 110-byte groups: the buffer ends mid-chunk
    (776, 7, 10, ["Q2_K", "Q6_K", "IQ3_S"]),  # 4 groups, a partial last workgroup
    (1280, 9, 7, ["Q3_K", "Q5_K"]),          # 5 groups: 3 rows, one slot over
    (4096, 3, 4, ["Q6_K", "Q4_K"]),          # 16 groups: one row
    (4360, 3, 5, ["Q3_K", "Q8_0"]),          # 18 groups: two segments of 9
])
def test_rows_sharing_a_workgroup(dim, vocab, nids, types):
    from voodoo_quant import _hip

    d_pad = (dim + 255) // 256 * 256
    g = torch.Generator().manual_seed(dim + nids)
    ids = torch.randint(0, vocab, (nids,), generator=g)
    ids[-1] = vocab - 1
    bad = torch.zeros(nids, dtype=torch.bool)
    if nids > 2:
        ids[1], bad[1] = vocab, True
        ids[2], bad[2] = -1, True
    qbs, cands = [], []
    for qt in types:
        nb = vocab * d_pad // 256 * (8 if qt == "Q8_0" else 1)
        q = torch.randint(0, 256, (nb, blocks.BLOCK_BYTES[qt]), dtype=torch.uint8, generator=g)
        for off in blocks.F16_OFFSETS[qt]:
            q[:, off + 1] = (q[:, off + 1] & 0x83) | 0x28
        qbs.append(q.reshape(-1).cuda())
        cands.append(torch.from_numpy(cdequant.oracle_dequant(qt, q.numpy(), vocab * d_pad).reshape(vocab, d_pad)))
    tids = [GGML[t] for t in types]
    probs = torch.softmax(torch.randn(len(types), generator=g), 0).cuda()
    safe = ids.clamp(0, vocab - 1)
    # the mixture: the same rows of W_eff, bit for bit
    w_eff = _hip.mix_weight(tids, qbs, probs, vocab, d_pad).cpu()
    want = w_eff[safe][:, :dim].clone()
    want[bad] = 0
    got = _hip.embedding_rows_fwd(tids, qbs, probs, None, ids.cuda(), vocab, dim, d_pad).cpu()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    # routed, fp32: the candidates' values, bit for bit; a route out of range gives a zero row
    route = torch.arange(nids) % len(types)
    if nids > 3:
        route[3] = len(types)
    zero = bad | (route >= len(types))
    want = torch.stack([cands[min(int(k), len(types) - 1)][i, :dim] for k, i in zip(route, safe)])
    want[zero] = 0
    got = _hip.embedding_rows_fwd(tids, qbs, None, route.cuda(), ids.cuda(), vocab, dim, d_pad, torch.float32).cpu()
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))
    # dL/dp: fp32 sums of at most 16 + 6 + 4 steps per workgroup, then fp64
    for dtype in (torch.bfloat16, torch.float32):
        dy = torch.randn(nids, dim, generator=g).to(dtype)
        terms = [(dy.double() * c[safe][:, :dim].double())[~bad] for c in cands]
        # the K-quant min and a code's offset are summed apart from the codes: up to twice the run's largest weight
        dp = _hip.embedding_rows_bwd(tids, qbs, ids.cuda(), vocab, dim, d_pad, dy.cuda()).double().cpu()
        for k, t in enumerate(terms):
            size = cands[k].abs().max().double() * dy.double().abs()[~bad].sum()
            assert (dp[k] - t.sum()).abs() <= 32 * 2.0**-24 * 4 * size + 2.0**-24 * t.sum().abs()


@pytest.mark.parametrize("n,at,value", [(1, 0, 10), (1, 0, 9), (8192, 8191, -1), (8193, 8192, 10), (20000, 9000, 1 << 40),
                                        (20000, 0, 0)])
def test_id_range_check(n, at, value):
    from voodoo_quant import _hip

    ids = torch.arange(n) % 10
    ids[at] = value
    assert bool(_hip.ids_out_of_range(ids.cuda(), 10)[0]) == (not 0 <= value < 10)
