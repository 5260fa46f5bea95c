"""Products of 17 to 128 rows through the ring in LDS: the plans on the host, the kernel at the edges of its tiles, chunks and
shares against float64, and rows whose results do not depend on the batch."""
import itertools

import pytest
import torch

from jax_vllm_amd.ops import kernels as K

from .test_kernels_gpu import gate_activation, randn

FORMS = list(itertools.product((32, 64, 128), (32, 64, 96, 128)))


def test_plans_are_ones_the_kernel_takes():
    for m, n, k, mode in itertools.product((16, 17, 32, 33, 64, 65, 128, 129), (4, 64, 1000, 1024, 4096, 5120, 6144, 24576, 51200, 151936),
                                           (32, 64, 128, 2048, 2080, 4096, 12288, 25600), ("parts", "rows", "pairs")):
        form = K.ring_plan(m, n, k, mode)
        if form is not None:
            assert 16 < m <= form[0] and form[:2] in FORMS and k % 64 == 0
            assert (2 <= form[2] <= min(4, k // 64)) if mode == "parts" else form[2] == 1
    assert K.ring_plan(64, 24576, 4096, "pairs") == (64, 96, 1)            # one block a compute unit
    assert K.ring_plan(64, 4096, 12288, "parts") == (64, 64, 4)
    assert K.ring_plan(24, 4096, 4096, "parts") is None                    # blocks that stay
    assert K.ring_plan(64, 51200, 5120, "pairs") is None                   # the library


def test_whole_inner_sizes_go_where_they_are_faster():
    """Blocks that take the whole inner size wait for their chunks, not for the memory, while w is small beside its inner size:
    there the library, which may share it out, was measured faster; and forms that leave compute units without a block lose."""
    for m, n, k in ((32, 4096, 3072), (24, 6144, 4096), (32, 8192, 5120), (17, 8192, 4096), (24, 10240, 4096), (24, 2080, 2048), (48, 6144, 4096),
                    (112, 3072, 1536), (24, 5120, 5120), (64, 2048, 4096)):
        assert K.ring_plan(m, n, k, "rows") is None, (m, n, k)
    for m, n, k, mode, tw in ((32, 16384, 4096, "pairs", 64), (24, 11296, 2048, "rows", 64), (64, 32000, 2048, "rows", 128), (72, 10240, 4096, "rows", 64),
                              (64, 151936, 4096, "rows", 128), (72, 8192, 1024, "rows", 32), (24, 24576, 4096, "pairs", 96)):
        form = K.ring_plan(m, n, k, mode)
        assert form is not None and form[1] == tw, (m, n, k, form)
    assert K.ring_plan(32, 8192, 4096, "parts") == (32, 128, 4) and K.ring_plan(32, 8192, 2048, "parts") == (32, 128, 4)
    assert K.ring_plan(40, 2560, 4096, "parts") is None                    # blocks that stay


@pytest.mark.gpu
@pytest.mark.parametrize("tm,tw", FORMS)
def test_products_at_the_edges(tm, tw):
    for m, n, k, parts in ((tm, tw, 64, 1), (tm - 15, tw + 4, 128, 2), (17, 3 * tw - 4, 64 * 11, 3), (tm, 2 * tw, 64 * 37, 4)):
        x, w = randn(m, k, dtype=torch.bfloat16, seed=m, scale=0.5), randn(n, k, dtype=torch.bfloat16, seed=n + k, scale=0.5)
        want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
        y = K.gemm_stream(x, w, (tm, tw, parts), "parts")
        assert y.shape == (parts, m, n)
        assert ((y.double().sum(0) - want).abs() <= 2.0 ** -24 * k * size).all()       # exact products, at most k float sums
        rows = K.gemm_stream(x, w, (tm, tw, 1))
        torch.testing.assert_close(rows.double(), want, rtol=2.0 ** -8, atol=2.0 ** -24 * k * float(size.max()))      # rounded once
        assert torch.equal(K.gemm_stream(x[:m // 2].contiguous(), w, (tm, tw, parts), "parts"), y[:, :m // 2])
        if n % 2 == 0:
            act = K.gemm_stream(x, w, (tm, tw, 1), "pairs", "silu")
            torch.testing.assert_close(act.double(), gate_activation("silu", want[:, 0::2]) * want[:, 1::2], rtol=1e-2, atol=1e-2)


@pytest.mark.gpu
def test_linear_takes_the_ring_and_refuses_what_it_must():
    x, w = randn(65, 2048, dtype=torch.bfloat16, seed=1, scale=0.5), randn(2048, 2048, dtype=torch.bfloat16, seed=2, scale=0.05)
    want = x.double() @ w.double().T
    assert K.linear(x, w, partial_ok=True).dim() == 3
    logits = K.linear(x, randn(8192, 2048, dtype=torch.bfloat16, seed=3), out_dtype=torch.float32)
    assert logits.dtype == torch.float32 and logits.shape == (65, 8192)
    for view in (x[:, :1024], randn(65 * 2048 + 1, dtype=torch.bfloat16, seed=4)[1:].view(65, 2048)):      # strided; 2 bytes off
        ww = w[:, :view.shape[1]].contiguous()
        got = K.linear(view, ww, partial_ok=True)
        assert got.dim() == 2                                             # the library's
        torch.testing.assert_close(got.double(), view.double() @ ww.double().T, rtol=2e-2, atol=5e-2)
    torch.testing.assert_close(K.linear(x, w, partial_ok=True).double().sum(0), want, rtol=1e-3, atol=1e-3)
    for args in (((32, 64, 1), "rows"), ((128, 48, 1), "rows"), ((128, 64, 2), "rows"), ((128, 64, 33), "parts")):
        with pytest.raises(K.KernelArgumentError):
            K.gemm_stream(x, w, *args)
    with pytest.raises(K.KernelArgumentError):
        K.gemm_stream(x[:, :2016].contiguous(), w[:, :2016].contiguous(), (128, 64, 1))      # the inner size no multiple of 64
