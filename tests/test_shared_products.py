"""Products of 129 to 1,024 rows whose inner size is shared out to blocks: the plans on the host, the kernel at the edges of its
tiles, of its ring and of its shares against float64."""
import itertools

import pytest
import torch

from jax_vllm_amd.ops import kernels as K

from .test_kernels_gpu import randn

TILES = ((128, 128), (256, 128), (256, 256))


def test_plans_are_ones_the_kernel_takes():
    for m, n, k in itertools.product((128, 129, 160, 300, 512, 1024, 1025, 2048), (4, 1000, 2080, 4096, 8192), (64, 128, 2048, 2080, 4096, 12288, 25600)):
        form = K.shares_plan(m, n, k)
        if form is not None:
            assert 128 < m <= 1024 and form[:2] in TILES and 2 <= form[2] <= min(4, k // 64) and k % 64 == 0
    assert K.shares_plan(160, 4096, 12288) == (128, 128, 4)
    assert K.shares_plan(512, 4096, 12288)[:2] == (256, 128)
    assert K.shares_plan(300, 4096, 4096) is not None
    assert K.shares_plan(2048, 4096, 4096) is None and K.shares_plan(300, 2048, 512) is None       # the library


def test_small_results_stay_with_the_library():
    """Measured faster there: 256 rows against 1,024 x 3,072 13.4 us with the norm that reads the result, 16.5 through partial sums."""
    for m, n, k in ((256, 1024, 3072), (200, 1024, 4096), (300, 768, 3072), (129, 768, 3072)):
        assert K.shares_plan(m, n, k) is None
    assert K.shares_plan(257, 1024, 3072) is not None and K.shares_plan(160, 2048, 4096) is not None


@pytest.mark.gpu
@pytest.mark.parametrize("tm,tw", TILES)
def test_products_at_the_edges(tm, tw):
    # chunks a part: 1, 2, 3, 4 (fewer than the ring holds), 5 and 6 (it turns once), 37 / 3
    for m, n, chunks, parts in ((tm, tw, 1, 1), (129, tw - 4, 2, 1), (tm + 1, 2 * tw, 5, 2), (2 * tm - 31, tw + 36, 4, 1), (tm - 1, tw, 10, 2),
                                (300, 260, 23, 4), (tm, 3 * tw, 37, 3)):
        k = chunks * 64
        x, w = randn(m, k, dtype=torch.bfloat16, seed=m, scale=0.5), randn(n, k, dtype=torch.bfloat16, seed=n + k, scale=0.5)
        want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
        y = K.gemm_shares(x, w, (tm, tw, parts))
        assert y.shape == (parts, m, n)
        assert ((y.double().sum(0) - want).abs() <= 2.0 ** -24 * k * size).all()       # exact products, at most k float sums


@pytest.mark.gpu
def test_linear_takes_the_shares_and_refuses_what_it_must():
    x, w = randn(160, 4096, dtype=torch.bfloat16, seed=1, scale=0.5), randn(4096, 4096, dtype=torch.bfloat16, seed=2, scale=0.05)
    want = x.double() @ w.double().T
    y = K.linear(x, w, partial_ok=True)
    assert y.dim() == 3 and y.dtype == torch.float32
    torch.testing.assert_close(y.double().sum(0), want, rtol=1e-3, atol=1e-3)
    assert K.linear(x, w).dim() == 2
    off = randn(160 * 4096 + 1, dtype=torch.bfloat16, seed=4)[1:].view(160, 4096)
    for view in (off, randn(160, 8192, dtype=torch.bfloat16, seed=5)[:, :4096]):           # 2 bytes off; strided
        got = K.linear(view, w, partial_ok=True)
        assert got.dim() == 2                                                              # the library's
        torch.testing.assert_close(got.double(), view.double() @ w.double().T, rtol=2e-2, atol=5e-2)
    for form in ((64, 128, 2), (128, 256, 2), (128, 128, 65)):
        with pytest.raises(K.KernelArgumentError):
            K.gemm_shares(x, w, form)
    with pytest.raises(K.KernelArgumentError):
        K.gemm_shares(x[:, :4064].contiguous(), w[:, :4064].contiguous(), (128, 128, 2))   # the inner size no multiple of 64
