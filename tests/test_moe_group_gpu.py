"""Groupings of (token, choice) entries that stay in registers or wait in memory."""
import pytest
import torch

from .test_kernels_gpu import K


@pytest.mark.gpu
@pytest.mark.parametrize("entries", [1, 4095, 4096, 4097, 8192, 8193, 16384, 16385])
@pytest.mark.parametrize("experts", [1, 7, 300])
def test_groupings(entries, experts):
    g = torch.Generator().manual_seed(entries)
    plan = K().moe_route(torch.randn(entries, experts, generator=g).cuda() if entries > 64 else torch.randn(65, experts, generator=g).cuda(), 1, tile_rows=64)
    ids, order, offsets = plan.ids.cpu(), plan.order.cpu().long(), plan.offsets.cpu()
    counts = torch.bincount(ids, minlength=experts)
    assert torch.equal(order.sort().values, torch.arange(ids.numel()))
    assert torch.equal(ids[order], ids.sort().values) and torch.equal(offsets.diff(), counts.int())
    tiles = int(plan.meta[0])
    assert tiles == int((-(-counts // 64)).sum())
    want = [(e, int(offsets[e]) + r) for e in range(experts) for r in range(0, int(counts[e]), 64)]
    assert list(zip(plan.tile_expert[:tiles].tolist(), plan.tile_row0[:tiles].tolist())) == want
