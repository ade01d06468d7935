"""vq_route_tokens against torch's stable sort: chunk edges of its one
workgroup, empty routes, every candidate count's ends, routes outside the
range, and the refusal of those in the routed forward."""

import pytest
import torch

from voodoo_quant import _hip, layers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 6, 16])
@pytest.mark.parametrize("m", [0, 1, 1023, 1024, 1025, 8192, 100003])
@pytest.mark.parametrize("stray", [False, True], ids=["valid", "stray"])
def test_grouping_is_a_stable_sort(m, k, stray):
    g = torch.Generator().manual_seed(m + k)
    routing = torch.randint(0, k, (m,), generator=g)
    if k > 2:
        routing[routing == 1] = 2  # an empty route
    if stray and m:
        routing[:: max(1, m // 7)] = torch.tensor([-1, k, 1 << 40, -(1 << 40)])[: 1 + m % 4].repeat(8)[: len(routing[:: max(1, m // 7)])]
    perm, plan = _hip.route_tokens(routing.cuda(), k)
    ok = (routing >= 0) & (routing < k)
    tokens = ok.nonzero().view(-1)
    want = tokens[torch.argsort(routing[ok], stable=True)]
    off = torch.zeros(k + 1, dtype=torch.int64)
    off[1:] = torch.cumsum(torch.bincount(routing[ok], minlength=k), 0)
    assert torch.equal(plan.cpu().long(), torch.cat([off, torch.tensor([m - int(ok.sum())])]))
    assert torch.equal(perm.cpu().long()[: len(want)], want)
    assert bool((perm.cpu()[len(want):] == -1).all())


@pytest.mark.parametrize("bad", [-1, 2])
def test_routed_forward_refuses_stray_routes(bad):
    m, n, d = 40, 64, 256
    cands = [torch.randn(n, d, device="cuda").bfloat16() for _ in range(2)]
    qbs = [torch.zeros(n * 272, dtype=torch.uint8, device="cuda") for _ in range(2)]
    routing = torch.zeros(m, dtype=torch.int64, device="cuda")
    routing[7] = bad
    with pytest.raises(RuntimeError):
        layers.RoutedLinearFunction.apply(torch.randn(m, d, device="cuda").bfloat16(),
                                          torch.full((2,), 0.5, device="cuda"), routing, ((8, 8), n, d), cands, *qbs)
