"""Expert products of few rows an expert with a ring a wave in LDS: every share of the inner size, odd numbers of chunks, rows of W that do
not fill a block, 0 to 17 rows an expert, against float64; operands and sizes that go the other way."""
import pytest
import torch

from .test_kernels_gpu import K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden,ff", [(64, 64), (448, 576), (704, 1024), (1088, 320), (2112, 136), (4096, 192), (40, 72), (4160, 64)])
@pytest.mark.parametrize("gated,on_input", [(True, True), (True, False), (False, False)])
def test_few_rows_an_expert(hidden, ff, gated, on_input):
    rows = [1, 0, 16, 17, 3]
    n, experts = sum(rows), len(rows)
    g = torch.Generator().manual_seed(hidden + ff)
    x = torch.randn(n, hidden, generator=g).bfloat16()
    wg, wu = ((torch.randn(experts, ff, hidden, generator=g) * hidden ** -0.5).bfloat16() for _ in range(2))
    wd = (torch.randn(experts, hidden, ff, generator=g) * ff ** -0.5).bfloat16()
    expert = torch.cat([torch.full((r,), e) for e, r in enumerate(rows)])[torch.randperm(n, generator=g)]
    logits = torch.full((n, experts), -4.0)
    logits[torch.arange(n), expert] = 1.0
    plan = K().moe_route(logits.cuda(), 1, tile_rows=16)
    out = torch.full((1, n, hidden), float("nan"), device="cuda")
    K().moe_experts(x.cuda(), plan, wg.cuda() if gated else None, wu.cuda(), wd.cuda(), "silu", out, weight_on_input=on_input)
    weight = torch.sigmoid(torch.tensor(1.0)).double()
    for e in range(experts):
        at = expert == e
        xs = x[at].double() * (weight if on_input else 1.0)
        u = xs @ wu[e].double().T
        h = xs @ wg[e].double().T if gated else u
        z = (h * torch.sigmoid(h) * (u if gated else 1.0)).bfloat16().double()      # what the kernels keep between the products
        want = (1.0 if on_input else weight) * z @ wd[e].double().T
        # z may be rounded the other way where the float sum and this one straddle: half a unit of bfloat16 in one term
        scale = z.abs() @ wd[e].double().abs().T + 1e-3
        assert ((out[0].cpu()[at].double() - want).abs() <= 2.0 ** -8 * scale).all()


def test_weights_off_16_bytes_go_the_other_way():
    n, experts, hidden, ff = 5, 3, 128, 192
    g = torch.Generator().manual_seed(5)
    x, wg, wu, wd = ((torch.randn(s, generator=g) * s[-1] ** -0.5).bfloat16().cuda() for s in ((n, hidden), (experts, ff, hidden), (experts, ff, hidden), (experts, hidden, ff)))
    off = torch.empty(wu.numel() + 1, dtype=torch.bfloat16, device="cuda")[1:].view(wu.shape).copy_(wu)
    plan = K().moe_route(torch.randn(n, experts, generator=g).cuda(), 2, tile_rows=16)
    results = []
    for up in (wu, off):
        out = torch.full((2, n, hidden), float("nan"), device="cuda")
        K().moe_experts(x, plan, wg, up, wd, "silu", out)
        results.append(out)
    torch.testing.assert_close(*results, rtol=2.0 ** -7, atol=1e-4)      # a rounding of z between the products


@pytest.mark.parametrize("n,experts,top,hidden", [(1, 32, 4, 2048), (16, 40, 3, 448), (7, 33, 4, 512)])
def test_router_logits_of_few_rows(n, experts, top, hidden):
    g = torch.Generator().manual_seed(n)
    x, wr = torch.randn(n, hidden, generator=g).bfloat16(), torch.randn(experts, hidden, generator=g).bfloat16()
    logits = torch.empty(n, experts, device="cuda")
    plan = K().moe_route(None, top, x=x.cuda(), w_router=wr.cuda(), logits_out=logits, tile_rows=16)
    want = x.double() @ wr.double().T
    assert ((logits.cpu().double() - want).abs() <= 2.0 ** -24 * hidden * (x.double().abs() @ wr.double().abs().T)).all()
    assert torch.equal(plan.ids.cpu().view(n, top).long().sort(-1).values, torch.topk(logits.cpu(), top).indices.sort(-1).values)
