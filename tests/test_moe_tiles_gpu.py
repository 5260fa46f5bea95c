"""The expert products' tiles and the router's logits at the edges of their tiles and chunks, against float64."""
import pytest
import torch

from .test_kernels_gpu import K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(1, 1, 8), (65, 15, 24), (79, 17, 256), (130, 33, 264), (300, 64, 2040), (81, 130, 520)])
def test_router_logits(m, n, k):
    g = torch.Generator().manual_seed(m)
    x, w = torch.randn(m, k, generator=g).bfloat16(), torch.randn(n, k, generator=g).bfloat16()
    y = K().gemm_rows_f32out(x.cuda(), w.cuda())
    # exact products, sums of k terms in float: well inside one rounding per term
    bound = 2.0 ** -24 * k * (x.double().abs() @ w.double().abs().T)
    assert ((y.cpu().double() - x.double() @ w.double().T).abs() <= bound).all()
    assert torch.equal(K().gemm_rows_f32out(x[m // 2:].contiguous().cuda(), w.cuda()), y[m // 2:])      # whatever the batch


@pytest.mark.parametrize("m,n,k,tiles", [(4096, 64, 1024, False), (4097, 64, 1024, True), (2050, 132, 2048, True), (1100, 516, 448, True),
                                         (8192, 32, 256, False), (1100, 513, 448, False), (1100, 516, 456, False)])
def test_router_logits_of_many_rows(m, n, k, tiles):
    """Beyond a round of blocks of 16 rows: tiles of 128 x 128, where the sizes allow them."""
    assert K().rows_by_tiles(m, n, k) == tiles
    g = torch.Generator(device="cuda").manual_seed(m)
    x, w = torch.randn(m, k, generator=g, device="cuda").bfloat16(), torch.randn(n, k, generator=g, device="cuda").bfloat16()
    y = K().gemm_rows_f32out(x, w)
    assert y.shape == (m, n) and y.dtype == torch.float32 and y.is_contiguous()
    bound = 2.0 ** -24 * k * (x.double().abs() @ w.double().abs().T)       # exact products, sums of k terms in float
    assert ((y.double() - x.double() @ w.double().T).abs() <= bound).all()


FEW = [40, 0, 1, 65, 17]           # 25 an expert: the form with two chunks on their way


def test_more_than_64_rows_an_expert_take_tiles_of_128():
    args = torch.bfloat16, 4096, 4096
    assert [K().moe_tile_rows_for(*args, n, 8) for n in (48, 49, 512, 513, 600)] == [16, 64, 64, 128, 128]
    assert K().moe_tile_rows_for(torch.float32, 4096, 4096, 600, 8) == 64


@pytest.mark.parametrize("tile_rows,few", [(64, False), (128, False), (64, True)])
@pytest.mark.parametrize("hidden,ff", [(8, 8), (56, 72), (64, 264), (136, 128), (200, 520)])
@pytest.mark.parametrize("gated", [True, False])
def test_expert_tiles(tile_rows, few, hidden, ff, gated):
    """Experts with no row, one row, a tile exactly, one more, and several tiles; one to nine chunks of the inner size."""
    rows = FEW if few else [tile_rows, 0, 1, tile_rows + 1, 2 * tile_rows + 33]
    n, experts = sum(rows), len(rows)
    g = torch.Generator().manual_seed(hidden + ff)
    x = torch.randn(n, hidden, generator=g).bfloat16()
    wg, wu = ((torch.randn(experts, ff, hidden, generator=g) * hidden ** -0.5).bfloat16() for _ in range(2))
    wd = (torch.randn(experts, hidden, ff, generator=g) * ff ** -0.5).bfloat16()
    expert = torch.cat([torch.full((r,), e) for e, r in enumerate(rows)])[torch.randperm(n, generator=g)]
    logits = torch.full((n, experts), -4.0)
    logits[torch.arange(n), expert] = 1.0
    plan = K().moe_route(logits.cuda(), 1, tile_rows=tile_rows)
    assert torch.equal(plan.ids.cpu().long(), expert)
    out = torch.full((1, n, hidden), float("nan"), device="cuda")
    K().moe_experts(x.cuda(), plan, wg.cuda() if gated else None, wu.cuda(), wd.cuda(), "silu", out, weight_on_input=False)
    weight = torch.sigmoid(torch.tensor(1.0)).double()
    for e in range(experts):
        at = expert == e
        u = x[at].double() @ wu[e].double().T
        h = x[at].double() @ wg[e].double().T if gated else u
        z = (h * torch.sigmoid(h) * (u if gated else 1.0)).bfloat16().double()      # what the kernels keep between the products
        want = weight * z @ wd[e].double().T
        # z may be rounded the other way where the float sum and this one straddle: half a unit of bfloat16 in one term
        scale = z.abs() @ wd[e].double().abs().T + 1e-3
        assert ((out[0].cpu()[at].double() - want).abs() <= 2.0 ** -8 * scale).all()


@pytest.mark.parametrize("which", [0, 1, 2, 3])
def test_an_operand_off_its_boundary(which):
    """Rows go into LDS in pieces of 16 bytes: an operand that begins 2 bytes off gives what its copy gives."""
    n, experts, hidden, ff = 150, 3, 72, 136
    g = torch.Generator().manual_seed(5)
    shapes = [(n, hidden), (experts, ff, hidden), (experts, ff, hidden), (experts, hidden, ff)]
    tensors = [(torch.randn(s, generator=g) * s[-1] ** -0.5).bfloat16().cuda() for s in shapes]
    off = list(tensors)
    flat = torch.empty(tensors[which].numel() + 1, dtype=torch.bfloat16, device="cuda")
    off[which] = flat[1:].view(shapes[which]).copy_(tensors[which])
    assert off[which].data_ptr() % 16 == 2 and off[which].is_contiguous()
    plan = K().moe_route(torch.randn(n, experts, generator=g).cuda(), 2, tile_rows=64)
    results = []
    for x, wg, wu, wd in (tensors, off):
        out = torch.full((2, n, hidden), float("nan"), device="cuda")
        K().moe_experts(x, plan, wg, wu, wd, "silu", out)
        results.append(out)
    assert torch.isfinite(results[0]).all() and torch.equal(*results)
