"""The 32-bit product on the bf16 matrix unit: every form of it to the bit, against float64, at the edges of tiles and steps; values
that are not finite or that no bf16 is near to."""
import pytest
import torch

from .test_kernels_gpu import K, randn

FORMS = range(11)


def product(form, a, w):
    """One form, whatever the plan would take (as ``gemm_f32`` launches it)."""
    k = K()
    plan = k.f32_plan
    try:
        k.f32_plan = lambda *_: form
        return k.gemm_f32(a, w)
    finally:
        k.f32_plan = plan


def bound(a, w):
    """A step's six products and their sum, the chain of a half's steps, the halves; what is dropped is below 2^-26 of the whole."""
    steps = -(-a.shape[1] // 32)
    return 2.0 ** -24 * (steps / 2 + 16) * (a.double().abs() @ w.double().abs().T)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(1, 1, 4), (16, 15, 32), (17, 33, 36), (33, 97, 64), (65, 130, 96), (129, 31, 100), (130, 260, 2048), (64, 64, 2080)])
def test_every_form_gives_the_same_bits(m, n, k):
    a, w = randn(m, k, seed=m), randn(n, k, seed=n + k)
    want = a.double() @ w.double().T
    outs = [product(form, a, w) for form in FORMS]
    assert ((outs[0].double() - want).abs() <= bound(a, w)).all()
    for form, out in zip(FORMS, outs):
        assert torch.equal(out, outs[0]), form


@pytest.mark.gpu
@pytest.mark.parametrize("m", [3, 40, 130])
@pytest.mark.parametrize("k", [1, 31, 127, 257])
def test_inner_sizes_and_addresses_without_pieces(m, k):
    """Rows that do not begin on 16 bytes: through registers, or w copied for tiles."""
    a, w = randn(m, k, seed=m), randn(70, k, seed=k)
    out = K().gemm_f32(a, w)
    assert ((out.double() - a.double() @ w.double().T).abs() <= bound(a, w)).all()
    for form in (0, 1, 5, 10):
        assert torch.equal(product(form, a, w), out), form
    off = torch.empty(70 * 64 + 1, device="cuda")[1:].view(70, 64)                 # w 4 bytes off
    off.copy_(randn(70, 64, seed=5))
    x = torch.empty(m * 64 + 1, device="cuda")[1:].view(m, 64)
    x.copy_(randn(m, 64, seed=6))
    assert torch.equal(K().gemm_f32(x, off), K().gemm_f32(x.clone(), off.clone()))


@pytest.mark.gpu
@pytest.mark.parametrize("k", [100, 256])
def test_values_that_the_split_does_not_hold(k):
    """Infinities and NaN as in 32-bit arithmetic; the largest floats (no bf16 is near to them) keep their products."""
    a, w = randn(40, k, seed=1), randn(70, k, seed=2)
    a[3, 5], a[7, k - 1], w[11, 9] = float("inf"), float("nan"), 0.0
    a[20, 9], w[2, 1] = 3.4e38, 3.4e38
    a[:, 1] *= 1e-3
    want = a.double() @ w.double().T
    want = torch.where(want.abs() > 3.4028235e38, want.sign() * float("inf"), want)      # beyond float: infinity, NaN stays
    for form in FORMS:
        out = product(form, a, w).double()
        assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out.isinf(), want.isinf()), form
        fine = want.isfinite()
        assert ((out - want).abs()[fine] <= (2.0 ** -24 * k * (a.double().abs() @ w.double().abs().T))[fine]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("ea,ew", [(-112, 0), (0, -118), (-126, 90), (80, -140), (-140, 20), (-60, -75), (100, -140), (30, 49)])
def test_numbers_at_the_ends_of_the_range_keep_their_bits(ea, ew):
    """Operands around 2^ea and 2^ew, subnormal ones among them, beside ones 2^20 larger and zeros: as exact as ordinary numbers, and a
    result below the smallest normal float within half a unit of its last place."""
    k = 160
    a, w = (randn(40, k, seed=1).double() * 2.0 ** ea).float(), (randn(70, k, seed=2).double() * 2.0 ** ew).float()
    a[:, ::7] *= 2.0 ** 20
    a[:, ::5], w[:, 1::9], a[11] = 0.0, 0.0, 0.0
    want = a.double() @ w.double().T
    outs = [product(form, a, w) for form in FORMS]
    assert (want.abs() > 2.0 ** -149).sum() > 1000      # something is left of them
    if ea > 80 or ea + ew > 50:      # beyond what the scaled split holds: one chain of k terms
        near = 2.0 ** -24 * k * (a.double().abs() @ w.double().abs().T)
    else:
        near = bound(a, w)
    assert ((outs[0].double() - want).abs() <= near + 2.0 ** -149).all()
    for form, out in zip(FORMS, outs):
        assert torch.equal(out, outs[0]), form


def test_every_size_has_a_form():
    from jax_vllm_amd.ops.kernels import KernelArgumentError, f32_plan

    for m in (1, 16, 17, 33, 64, 65, 300, 5000, 1 << 20):
        for n in (1, 31, 4096, 151936):
            for k in (0, 1, 32, 4096, 1 << 21):
                for pieces in (True, False):
                    form = f32_plan(m, n, k, pieces, pieces)
                    assert form in FORMS and (form < 5 or m > 32) and (form not in (2, 3, 4) or pieces)
                    assert form not in (2, 3, 4) or k > 0
    with pytest.raises(KernelArgumentError):
        f32_plan(1 << 30, 1 << 30, 32)


def test_forms_whose_blocks_go_two_to_a_unit():
    """From 257 blocks of 32 x 16 on a unit has two of them and takes as long as all do: these sizes take 8 to 18 % longer that way."""
    from jax_vllm_amd.ops.kernels import f32_plan

    for m, n, k in [(48, 3072, 2048), (80, 2048, 2048), (160, 1000, 4096), (333, 512, 4096), (32, 6144, 8192), (17, 6144, 8192), (24, 6144, 8192)]:
        assert f32_plan(m, n, k) == 4, (m, n, k)
    assert f32_plan(10, 4096, 6144) == f32_plan(10, 4096, 3072) == 2 and f32_plan(16, 32000, 2048) == f32_plan(24, 3072, 2048) == 3
