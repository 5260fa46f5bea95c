"""Which product reads rows whose norm's scale is still to be applied, on both sides of the lines where small blocks take over."""
import pytest

from .test_kernels_gpu import K, randn
from .test_thin_products import test_rows_with_many_shares_of_their_scale as product


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,pairs,thin", [
    (8, 6144, 3136, False, True), (9, 6144, 3072, False, True), (9, 6144, 3136, False, True), (9, 16388, 2624, False, False), (9, 24576, 2624, False, True), (16, 8192, 4096, False, True),
    (1, 8196, 2560, False, True), (8, 8200, 2624, False, False), (16, 16384, 64, True, True), (3, 12288, 2624, True, True)])
def test_lines_between_the_forms(m, n, k, pairs, thin):
    from jax_vllm_amd.ops import kernels

    assert (kernels._stream_rows_plan(m, randn(n, k, seed=1).bfloat16(), pairs, not pairs, None) == "thin") == thin
    product(m, n, k, pairs)


@pytest.mark.gpu
def test_a_whole_inner_size_by_blocks_that_stay_is_one_part():
    """A reader of partial products gets [1, M, N], also where blocks that stay hold the whole inner size (a q/k/v product of 16,388 columns)."""
    test_lines_between_the_forms(8, 16388, 512, False, False)
    w = randn(16388, 512, seed=1).bfloat16()
    rows = K().StreamRows(randn(8, 512, seed=2).bfloat16(), randn(8, 256, seed=3) ** 2, 512, 1e-6)
    assert K().linear(rows, w, partial_ok=True, partial_max_width=None).shape == (1, 8, 16388)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,pairs", [(1, 24576, 2624, True), (8, 24576, 1088, True), (8, 20484, 4032, False), (3, 20484, 1024, False)])
def test_blocks_that_stay_with_many_shares(m, n, k, pairs):
    """The form with 256 shares a row, inner sizes with and without a last piece beside the rows' end."""
    test_lines_between_the_forms(m, n, k, pairs, False)


@pytest.mark.gpu
def test_many_shares_where_no_reader_asks_for_them():
    """Rows with 256 shares go into float sums and activations of inner sizes up to 4,096: anything else is refused, not scaled by 16 of them."""
    w, x = randn(64, 1024, seed=1).bfloat16(), randn(2, 1024, seed=2).bfloat16()
    rows = K().StreamRows(x, randn(2, 256, seed=3) ** 2, 1024, 1e-6)
    with pytest.raises(K().KernelArgumentError):
        K().gemm_skinny(x, w, block_shape=(-2, 256, 4), row_scale=rows)
