"""Products of up to 16 rows with the inner size shared out to a block's waves: every output form at odd numbers of rows, chunks and
rows of W, against float64, and where they are taken."""
import pytest
import torch

from .test_kernels_gpu import K, randn


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 5, 15, 16])
@pytest.mark.parametrize("n,k", [(4, 64), (20, 448), (36, 512), (100, 576), (1028, 1088), (64, 2048), (48, 2112), (4100, 4096)])
@pytest.mark.parametrize("tile", [16, 32])
def test_few_rows(m, n, k, tile):
    x, w = randn(m, k, seed=m).bfloat16(), randn(n, k, seed=n + k).bfloat16()
    want = x.double() @ w.double().T
    y = K().gemm_few(x, w, tile, out_dtype=torch.float32)
    # exact products, eight chains of k / 8 terms and eight sums in float
    bound = 2.0 ** -24 * (k / 8 + 8) * (x.double().abs() @ w.double().abs().T)
    assert ((y.double() - want).abs() <= bound).all()
    assert torch.equal(K().gemm_few(x, w, tile), y.bfloat16())
    assert torch.equal(K().gemm_few(x[m // 2:].contiguous(), w, tile, out_dtype=torch.float32), y[m // 2:])      # whatever the batch
    gated = K().gemm_few(x, w, tile, "silu")
    g, u = y[:, 0::2], y[:, 1::2]
    torch.testing.assert_close(gated, (g / (1 + torch.exp(-g)) * u).bfloat16(), rtol=2.0 ** -7, atol=1e-6)      # a rounding of bfloat16


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(1, 5120, 1024), (4, 4100, 64), (3, 8192, 448), (9, 5120, 1024), (16, 6144, 576), (8, 8196, 1024), (16, 12288, 512), (1, 512, 768),
                                   (2, 1024, 1024)])
@pytest.mark.parametrize("tile", [16, 32])
def test_what_blocks_with_x_in_registers_take(m, n, k, tile):
    """The sizes that the rule leaves to them, and the bits of small blocks."""
    assert K().thin_slots(m, n, k) is None and K().few_tile(m, n, k) is not None
    test_few_rows(m, n, k, tile)


@pytest.mark.gpu
def test_given_rows_of_more_columns_are_refused(monkeypatch):
    monkeypatch.setattr(K(), "thin_slots", lambda *_: None)
    with pytest.raises(K().KernelArgumentError):
        K().gemm_few(randn(2, 1088, seed=1).bfloat16(), randn(64, 1088, seed=2).bfloat16(), 16)


@pytest.mark.gpu
def test_rows_that_are_not_finite_stay_alone():
    x, w = randn(9, 512, seed=1).bfloat16(), randn(64, 512, seed=2).bfloat16()
    clean = K().gemm_few(x, w, 16)
    x[4, 100], w[33, 7] = float("nan"), float("inf")
    y = K().gemm_few(x, w, 16)
    rows, cols = torch.arange(9) != 4, torch.arange(64) != 33
    assert torch.equal(y[rows][:, cols], clean[rows][:, cols]) and not y[4].isfinite().any() and not y[:, 33].isfinite().any()


@pytest.mark.gpu
def test_operands_the_form_does_not_take_go_the_old_way(monkeypatch):
    x, w = randn(6, 2048, seed=1).bfloat16(), randn(2048, 2048, seed=2).bfloat16()
    off = [torch.empty(t.numel() + 4, dtype=torch.bfloat16, device="cuda")[4:].view(t.shape).copy_(t) for t in (x, w)]
    assert all(t.data_ptr() % 16 == 8 and t.is_contiguous() for t in off)      # 8 bytes off

    def taken(*_, **__):
        raise AssertionError("operands that the form does not take")

    want = x.double() @ w.double().T
    with monkeypatch.context() as patch:
        patch.setattr(K(), "gemm_few", taken)
        for operands in ((off[0], w), (x, off[1])):
            y = K().linear(*operands)
            # a rounding to bfloat16 of a float sum of 2,048 products
            assert ((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -24 * 2048 * (x.double().abs() @ w.double().abs().T)).all()
        with pytest.raises(AssertionError, match="does not take"):
            K().linear(x, w)      # (aligned: it would be)
    assert K().few_tile(6, 2048, 2040) is None and K().few_tile(6, 2048, 4160) is None and K().few_tile(17, 2048, 2048) is None
    torch.testing.assert_close(K().linear(x[:, :2040].contiguous(), w[:, :2040].contiguous()).double(),
                               x[:, :2040].double() @ w[:, :2040].double().T, rtol=2.0 ** -7, atol=0.05)


def test_rows_of_w_of_a_block():
    from jax_vllm_amd.ops.kernels import STAGED, few_tile, streaming_plan

    assert [few_tile(8, n, 2048) for n in (32, 4096, 4112, 6144, 6160, 11296)] == [16, 16, 32, 32, 16, 16]
    assert streaming_plan(8, 6144, 2048, True) == STAGED and streaming_plan(12, 12288, 4096) is None


@pytest.mark.parametrize("m,n,k,partial_ok", [(4, 2048, 2048, False), (1, 151936, 4096, False), (12, 12288, 4096, False), (3, 96, 512, True), (16, 32, 512, False)])
def test_rows_without_their_scale_are_refused(monkeypatch, m, n, k, partial_ok):
    """Only blocks that stay multiply a row by its norm's scale: every other plan says so instead of leaving the scale out."""
    from jax_vllm_amd.ops import kernels

    def launched(*_, **__):
        raise AssertionError("a product of rows whose scale is still to be applied")

    monkeypatch.setattr(kernels, "compute_units", lambda device: 256)
    for name in ("gemm_few", "gemm_skinny", "gemm_stream", "gemm_tile64", "gemm_shares"):
        monkeypatch.setattr(kernels, name, launched)
    x, w = torch.zeros(m, k, dtype=torch.bfloat16), torch.empty(n, k, dtype=torch.bfloat16)      # (never read)
    rows = kernels.UnscaledRows(x, torch.ones(m, kernels.UNSCALED_MAX_SHARES), k, 1e-6)
    assert not kernels.linear_takes_unscaled_rows(m, w, partial_ok=partial_ok)
    with pytest.raises(kernels.KernelArgumentError, match="un-normalised rows"):
        kernels.linear(rows, w, partial_ok=partial_ok)


def test_one_row_against_the_output_embedding_stays_with_x_resident():
    from jax_vllm_amd.ops.kernels import STAGED, few_tile, streaming_plan

    assert streaming_plan(1, 151936, 4096) == streaming_plan(2, 151936, 4096) == STAGED      # the kernel library's choice: x resident
    assert [few_tile(m, n, k) for m, n, k in ((1, 151936, 4096), (1, 65536, 3584), (2, 151936, 4096), (1, 151936, 3328), (1, 151936, 2048), (1, 16000, 4096))] \
        == [None, None, 16, 16, 16, 16]


def test_rows_of_w_of_a_block_where_the_library_was():
    from jax_vllm_amd.ops.kernels import few_tile, streaming_plan, thin_slots, thin_tiles

    sizes = ((16, 15360, 4096), (9, 12304, 1536), (16, 12288, 4096), (8, 15360, 4096), (16, 15360, 1024))
    assert streaming_plan(16, 15360, 4096) is None and [few_tile(*s) for s in sizes] == [16] * 5
    # the tiles of a block are those of the small blocks here
    assert [thin_slots(*s) and thin_tiles(*s[:2]) for s in sizes] == [2, 2, 1, 1, None]
