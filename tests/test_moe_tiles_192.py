"""Expert products by tiles of 192 rows: at the ends of tiles, the same bits as by tiles of 128, and where they are chosen."""
import pytest
import torch

from .test_kernels_gpu import K


@pytest.mark.gpu
@pytest.mark.parametrize("hidden,ff", [(8, 8), (72, 136), (264, 520)])
@pytest.mark.parametrize("gated", [True, False])
def test_expert_tiles_of_192(hidden, ff, gated):
    """No row, one, 63 to 65 and 128 of a tile's 192 (its waves' tiles), a tile exactly, one more, several."""
    rows = [192, 0, 1, 193, 65, 128, 2 * 192 + 97]
    n, experts = sum(rows), len(rows)
    g = torch.Generator().manual_seed(hidden + ff)
    x = torch.randn(n, hidden, generator=g).bfloat16().cuda()
    wg, wu = ((torch.randn(experts, ff, hidden, generator=g) * hidden ** -0.5).bfloat16().cuda() for _ in range(2))
    wd = (torch.randn(experts, hidden, ff, generator=g) * ff ** -0.5).bfloat16().cuda()
    expert = torch.cat([torch.full((r,), e) for e, r in enumerate(rows)])[torch.randperm(n, generator=g)]
    logits = torch.full((n, experts), -4.0)
    logits[torch.arange(n), expert] = 1.0
    results = []
    for tile_rows in (128, 192):
        plan = K().moe_route(logits.cuda(), 1, tile_rows=tile_rows)
        out = torch.full((1, n, hidden), float("nan"), device="cuda")
        K().moe_experts(x, plan, wg if gated else None, wu, wd, "silu", out, weight_on_input=False)
        results.append(out)
    assert torch.isfinite(results[0]).all() and torch.equal(*results)      # (those of 128 are held against float64 beside)


def test_where_tiles_of_192_are_chosen():
    from jax_vllm_amd.ops.kernels import moe_tile_rows_for

    def rows(tokens, experts, top, hidden, ff):
        return moe_tile_rows_for(torch.bfloat16, hidden, ff, tokens * top, experts)

    assert [rows(n, 32, 4, 2048, 512) for n in (2048, 1500, 1024, 512)] == [192, 128, 128, 64]
    assert [rows(n, 64, 8, 2048, 1024) for n in (4096, 2048)] == [192, 192]
    assert [rows(n, 32, 4, 2048, 768) for n in (4096, 2048)] == [192, 128]
    assert moe_tile_rows_for(torch.float32, 2048, 512, 8192, 32) == 64
