"""Products of 1,025 to 1,792 rows by halves of a long inner size: which sizes take them, and the tiles of 192 x 256 at their edges."""
import itertools

import pytest
import torch

from jax_vllm_amd.ops import kernels as K


def test_one_round_that_fills_the_units():
    for m, n, k in itertools.product((1024, 1025, 1152, 1153, 1536, 1537, 1792, 1793, 2048), (4, 1024, 3000, 4096, 5120, 8192, 8190), (64, 4096, 8192, 8224, 12288, 25600)):
        form = K.tall_shares_plan(m, n, k)
        if form is not None:
            assert K.shares_plan(m, n, k) is None and 1024 < m <= 1792 and k >= 8192 and k % 64 == 0 and n % 4 == 0
            assert 192 <= -(-m // form[0]) * -(-n // form[1]) * form[2] <= 256
    assert [K.tall_shares_plan(m, 4096, 12288) for m in (1024, 1025, 1536, 1537, 1792, 1793)] == [None, *[(192, 256, 2)] * 2, *[(256, 256, 2)] * 2, None]
    assert K.tall_shares_plan(1300, 5120, 8192) is None and K.tall_shares_plan(1300, 5120, 17408) == (256, 256, 2)
    assert K.tall_shares_plan(1525, 1024, 12288) is None and K.tall_shares_plan(1525, 4096, 4096) is None


def numbers(m, n, k):
    g = torch.Generator().manual_seed(m + n + k)
    return ((torch.randn(s, k, generator=g) * 0.5).bfloat16().cuda() for s in (m, n))


@pytest.mark.gpu
# chunks a part: 1 to 4 (fewer than the ring holds), 5 and 6 (it turns once), 23 / 4
@pytest.mark.parametrize("m,n,chunks,parts", [(192, 256, 1, 1), (129, 252, 2, 1), (193, 512, 5, 2), (353, 292, 4, 1), (191, 256, 10, 2), (300, 260, 23, 4), (192, 768, 12, 2)])
def test_tiles_of_192_by_256(m, n, chunks, parts):
    x, w = numbers(m, n, chunks * 64)
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    y = K.gemm_shares(x, w, (192, 256, parts))
    assert y.shape == (parts, m, n)
    assert ((y.double().sum(0) - want).abs() <= 2.0 ** -24 * chunks * 64 * size).all()       # exact products, at most k float sums


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1025, 1700])
def test_linear_takes_them_where_parts_are_added(m):
    x, w = numbers(m, 4096, 8192 if m == 1025 else 12288)
    y = K.linear(x, w, partial_ok=True)
    assert y.shape == (2, m, 4096) and K.linear(x, w).dim() == 2
    want = x.double() @ w.double().T
    assert ((y.double().sum(0) - want).norm() <= 1e-5 * want.norm())
