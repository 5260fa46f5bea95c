"""Results of the grouped expert products that leave in whole pieces of four columns, and where the result does not begin on 16 bytes."""
import pytest
import torch

from .test_kernels_gpu import K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile_rows", [64, 128, 192])
@pytest.mark.parametrize("hidden,ff", [(136, 72), (320, 264), (256, 256)])
def test_results_off_16_bytes(tile_rows, hidden, ff):
    """Columns that end inside a block's and inside a wave's share; the last tile of an expert short by 1 to 63 rows."""
    n, experts, top = 211, 3, 2
    g = torch.Generator().manual_seed(hidden + tile_rows)
    x, wg, wu, wd = ((torch.randn(s, generator=g) * s[-1] ** -0.5).bfloat16().cuda() for s in ((n, hidden), (experts, ff, hidden), (experts, ff, hidden), (experts, hidden, ff)))
    plan = K().moe_route(torch.randn(n, experts, generator=g).cuda(), top, tile_rows=tile_rows)
    room, results = torch.full((top * n * hidden + 1,), float("nan"), device="cuda"), []
    for out in (torch.full((top, n, hidden), float("nan"), device="cuda"), room[1:].view(top, n, hidden)):
        K().moe_experts(x, plan, wg, wu, wd, "silu", out)
        results.append(out)
    assert torch.equal(*results) and not results[0].isnan().any() and room[0].isnan()
