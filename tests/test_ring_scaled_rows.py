"""Products of 17 to 128 rows whose norm's scale is still to be applied, in every output form, against float64."""
import pytest
import torch

from .test_kernels_gpu import K, randn


@pytest.mark.gpu
@pytest.mark.parametrize("m", [17, 32, 33, 64, 65, 128])
@pytest.mark.parametrize("n,k,how,tw,parts", [(6144, 1024, "parts", 64, 4), (100, 8192, "parts", 32, 3), (2048, 1024, "pairs", 96, 1), (516, 512, "rows", 128, 1)])
def test_scaled_rows(m, n, k, how, tw, parts):
    k_ = K()
    h, added, weight = randn(m, k, seed=m, scale=2.0), randn(3, m, k, seed=m + 1), 1 + 0.1 * randn(k, seed=2)
    v = h.double() + added.double().sum(0)
    rows = k_.add_parts_unscaled(h, added, weight, 1e-5)
    w = randn(n, k, dtype=torch.bfloat16, seed=n, scale=k ** -0.5)
    y = k_.gemm_stream(rows.x, w, (32 if m <= 32 else 64 if m <= 64 else 128, tw, parts), how, "silu" if how == "pairs" else None, row_scale=rows)
    z = rows.x.double() @ w.double().T * torch.rsqrt(v.square().mean(1, keepdim=True) + 1e-5)
    if how == "pairs":
        g, u = z[:, 0::2], z[:, 1::2]
        torch.testing.assert_close(y.double(), g / (1 + torch.exp(-g)) * u, rtol=2.0 ** -7, atol=1e-4)      # a rounding of bfloat16
    elif how == "rows":
        torch.testing.assert_close(y.double(), z, rtol=2.0 ** -8, atol=1e-4)
    else:
        assert y.dim() == 3
        # exact products and sums of k terms in float, the scale's sums and root
        bound = 2.0 ** -24 * (2 * k + 16) * (rows.x.double().abs() @ w.double().abs().T) * torch.rsqrt(v.square().mean(1, keepdim=True) + 1e-5)
        assert ((y.double().sum(0) - z).abs() <= bound).all()


@pytest.mark.gpu
def test_rows_that_do_not_belong_together_are_refused():
    k_ = K()
    rows = k_.add_parts_unscaled(randn(40, 1024, seed=1), randn(2, 40, 1024, seed=2), randn(1024, seed=3), 1e-5)
    w = randn(6144, 1024, dtype=torch.bfloat16, seed=4)
    with pytest.raises(k_.KernelArgumentError, match="does not belong"):
        k_.gemm_stream(rows.x.clone(), w, (64, 64, 1), "rows", row_scale=rows)
    assert torch.equal(k_.linear(rows, w, partial_ok=True), k_.gemm_stream(rows.x, w, k_.ring_plan(40, 6144, 1024, "parts"), "parts", row_scale=rows))
    assert k_.linear_takes_unscaled_rows(40, w, partial_ok=True) and not k_.linear_takes_unscaled_rows(129, w, partial_ok=True) and not k_.linear_takes_unscaled_rows(40, w[:, :1000].contiguous(), partial_ok=True)
