"""The order in which a decode attention's blocks take their requests: the device's ranking against the host's, and the same results in any order."""
import math

import pytest
import torch

from .test_kernels_gpu import K, randn


def places(n, at_once):
    """The rank (0: the longest) of the request at each place: the units that get a second request begin with the shorter of the first lap."""
    second = n - at_once
    if second <= 0:
        return list(range(n))
    if n <= 2 * at_once:
        return list(range(at_once - second, at_once)) + list(range(at_once - second)) + list(range(n - 1, at_once - 1, -1))
    order = []
    for lap, first in enumerate(range(0, n, at_once)):
        ranks = list(range(first, min(n, first + at_once)))
        order += ranks[::-1] if lap & 1 else ranks
    return order


@pytest.mark.parametrize("n,at_once", [(33, 32), (40, 32), (63, 32), (64, 32), (5, 3)])
def test_two_a_unit_share_evenly(n, at_once):
    order = places(n, at_once)
    assert sorted(order) == list(range(n))
    sums = {order[j] + order[j + at_once] for j in range(n - at_once)}
    assert len(sums) == 1 and sorted(order[n - at_once:at_once]) == list(range(2 * at_once - n))      # who is alone is among the longest


@pytest.mark.gpu
@pytest.mark.parametrize("window", [0, 300, -128])
@pytest.mark.parametrize("n,at_once", [(1, 1), (2, 1), (31, 32), (33, 32), (40, 32), (64, 32), (97, 32), (257, 64), (1024, 256), (1022, 7)])
def test_order_on_the_device(n, at_once, window):
    lens = torch.randint(0, 700 if n < 64 else 90, (n,), generator=torch.Generator().manual_seed(n), dtype=torch.int32)      # equal ones among them
    seen = [min(v, window) if window > 0 else v % -window if window < 0 else v for v in lens.tolist()]
    ranked = sorted(range(n), key=lambda i: (-seen[i], i))
    assert K().decode_order(lens.cuda(), at_once, window).tolist() == [ranked[q] for q in places(n, at_once)]


@pytest.mark.gpu
def test_results_do_not_depend_on_it():
    k_, n, nq, nkv, d, page = K(), 35, 16, 8, 128, 16
    lens = [(37 * i) % 601 for i in range(n)]
    pages = [c // page + 1 for c in lens]
    tables = torch.zeros(n, max(pages), dtype=torch.int32)
    at = 1
    for i, m in enumerate(pages):
        tables[i, :m] = torch.arange(at, at + m)
        at += m
    slots = torch.tensor([int(tables[i, c // page]) * page + c % page for i, c in enumerate(lens)], dtype=torch.int32).cuda()
    kp, vp = randn(at, nkv, page, d, dtype=torch.bfloat16, seed=1), randn(at, nkv, d, page, dtype=torch.bfloat16, seed=2)
    qkv, tables, ctx = randn(n, (nq + 2 * nkv) * d, dtype=torch.bfloat16, seed=3), tables.cuda(), torch.tensor(lens, dtype=torch.int32).cuda()
    cu = torch.arange(n + 1, dtype=torch.int32).cuda()
    order, results = k_.decode_order(ctx, 32), []
    for work in (None, order, order.flip(0).contiguous()):
        k, v, out = kp.clone(), vp.clone(), torch.zeros(n, nq * d, dtype=torch.bfloat16, device="cuda")
        k_.attn_decode_token(out, qkv, slots, None, None, 0.0, None, 0, k, v, tables, ctx, nq, nkv, d, 1 / math.sqrt(d), work=work)
        ready = torch.zeros_like(out)
        k_.attn_decode_mfma(ready, qkv, (nq + 2 * nkv) * d, k, v, tables, cu, ctx, work, n, nq, nkv, d, 1 / math.sqrt(d))
        results.append((out, ready, k, v))
    for other in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(results[0], other))
    with pytest.raises(k_.KernelArgumentError):
        k_.decode_order(torch.zeros(1025, dtype=torch.int32, device="cuda"), 32)
