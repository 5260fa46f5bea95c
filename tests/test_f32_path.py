"""The 32-bit path's products on the matrix cores: against float64 at the edges of tiles and parts, and bit by bit across
batches."""
import pytest
import torch

from .test_kernels_gpu import K, randn


# ------------------------------------------------------------------ matrix products
@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 15, 16, 17, 32, 33, 63, 65, 127, 129])
@pytest.mark.parametrize("n,k", [(1, 1), (15, 127), (16, 128), (33, 129), (63, 2047), (4099, 516), (8200, 144)])
def test_gemm_f32_tiles_and_parts(m, n, k):
    a, w = randn(m, k, seed=m), randn(n, k, seed=n + k)
    out = K().gemm_f32(a, w)
    want = a.double() @ w.double().T
    # eight chains of at most k / 8 + 16 fused steps and eight sums: far inside the bound of one chain of k
    assert ((out.double() - want).abs() <= 2.0 ** -24 * (k / 8 + 24) * (a.double().abs() @ w.double().abs().T)).all()
    # whatever tile the batch takes, a row's bits are the same
    for rows in (slice(0, 1), slice(m // 2, m // 2 + 1), slice(0, (m + 1) // 2)):
        assert torch.equal(K().gemm_f32(a[rows].contiguous(), w), out[rows])
