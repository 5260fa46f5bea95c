"""The 32-bit product: tiles of 128 rows at their edges, and the activation of pairs of rows of W as an epilogue of every form."""
import pytest
import torch

from .test_f32_split import FORMS, bound, product
from .test_kernels_gpu import K, randn


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(127, 191, 33 * 32), (128, 192, 64), (257, 129, 96), (160, 386, 2080), (33, 64, 32), (300, 1000, 700)])
def test_tiles_of_128_rows(m, n, k):
    a, w = randn(m, k, seed=m), randn(n, k, seed=n + k)
    few = product(4, a, w)
    assert ((few.double() - a.double() @ w.double().T).abs() <= bound(a, w)).all()
    for form in (5, 6, 7):
        assert torch.equal(product(form, a, w), few), form


@pytest.mark.gpu
@pytest.mark.parametrize("activation", ["silu", "gelu_tanh", ("clamped", 2.0, 1.7)])
@pytest.mark.parametrize("m,n,k", [(1, 2, 4), (5, 98, 64), (40, 130, 100), (130, 200, 96)])
def test_activation_as_an_epilogue(m, n, k, activation):
    """Bit for bit the product and then the activation, in every form; values the split does not hold among them."""
    a, w = randn(m, k, seed=m), randn(n, k, seed=n)
    if m > 1:
        a[0, 0] = 3.0e38
        a[m - 1, 1] = float("inf")
    k_ = K()
    plan = k_.f32_plan
    try:
        for form in FORMS:
            k_.f32_plan = lambda *_: form
            got = k_.gemm_f32(a, w, gate_pairs=activation)
            want = k_.gated_mul(k_.gemm_f32(a, w), interleaved=True, activation=activation)
            assert got.shape == (m, n // 2)
            assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num()), form
    finally:
        k_.f32_plan = plan
    out = torch.empty(m, n // 2, device="cuda")
    assert k_.linear(a, w, gate_pairs=activation).shape == out.shape and k_.gemm_f32(a, w, out, activation) is out
    with pytest.raises(k_.KernelArgumentError, match="pairs"):
        k_.gemm_f32(a, w[:n - 1], gate_pairs=activation)


@pytest.mark.gpu
def test_the_longest_rows():
    """Every inner size that a plan gives to the tiles: 65,536 blocks of columns split a row of 2^22."""
    k = 1 << 22
    assert K().f32_plan(500, 4096, k) == 7 and K().f32_plan(1024, 4096, k) == 5
    a, w = randn(33, k, seed=1), randn(2, k, seed=2)
    few = product(10, a, w)
    assert ((few.double() - a.double() @ w.double().T).abs() <= bound(a, w)).all()
    for form in (5, 6, 7):
        assert torch.equal(product(form, a, w), few), form
