"""Products of 9 to 16 rows by blocks of two tiles of W: the bits of one tile a block, and the sizes where the rule changes sides."""
import pytest
import torch

from .test_kernels_gpu import K, randn


@pytest.mark.gpu
@pytest.mark.parametrize("m", [9, 16])
@pytest.mark.parametrize("n,k", [(4100, 1088), (6144, 4096), (8192, 64), (16388, 1152)])
@pytest.mark.parametrize("form", ["bf16", "float", "pairs"])
def test_the_bits_of_one_tile_a_block(monkeypatch, m, n, k, form):
    x, w = randn(m, k, seed=m).bfloat16(), randn(n, k, seed=n).bfloat16()
    args = dict(gate_pairs="silu") if form == "pairs" else dict(out_dtype=torch.float32 if form == "float" else torch.bfloat16)
    monkeypatch.setattr(K(), "thin_slots", lambda *_: 2)
    monkeypatch.setattr(K(), "thin_tiles", lambda *_: 2)
    y = K().gemm_few(x, w, 16, **args)
    monkeypatch.setattr(K(), "thin_tiles", lambda *_: 1)
    assert torch.equal(y, K().gemm_few(x, w, 16, **args))
    rows = K().StreamRows(x, torch.rand(m, 256, device="cuda") + 0.1, k, 1e-6)
    one = K().gemm_thin_scaled(rows, w, args.get("gate_pairs"))
    monkeypatch.setattr(K(), "thin_tiles", lambda *_: 2)
    assert torch.equal(one, K().gemm_thin_scaled(rows, w, args.get("gate_pairs")))


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,partial", [(9, 6144, 4096, True), (16, 6146, 2048, True), (12, 24576, 2048, False), (16, 32000, 1088, False), (9, 12288, 2048, False)])
def test_linear_around_the_rule(m, n, k, partial):
    x, w = randn(m, k, seed=3).bfloat16(), randn(n, k, seed=4).bfloat16()
    y = K().linear(x, w, partial_ok=partial, partial_max_width=None)
    y = y.sum(0) if y.dim() == 3 else y
    z = x.double() @ w.double().T
    # a sum of k products in float in any order, and a rounding of bfloat16
    assert ((y.double() - z).abs() <= 2.0 ** -24 * k * (x.double().abs() @ w.double().abs().T) + 2.0 ** -8 * z.abs()).all()


def test_where_two_tiles_are_taken():
    from jax_vllm_amd.ops import kernels

    assert [kernels.thin_tiles(16, n) for n in (4096, 4100, 8192, 8196, 12288, 12292, 16384, 16388, 24576)] == [1, 2, 2, 1, 1, 2, 2, 1, 2]
    assert kernels.thin_tiles(8, 8192) == 1 and kernels.thin_tiles_pay(9, 8192, 2048) and not kernels.thin_tiles_pay(9, 8192, 1024)
    assert not kernels.thin_tiles_pay(9, 151936, 2048) and kernels.thin_tiles_pay(9, 151936, 4096)


def test_where_two_tiles_do_not_pay():
    from jax_vllm_amd.ops.kernels import thin_tiles_pay as pays

    assert [pays(16, 16384, k) for k in (1024, 1088, 2560, 3072, 4096)] == [False, True, True, True, True]
    for n in (24576, 32000):      # 7 to 10 pieces a wave of the blocks that stay, and 12 whole ones
        assert [pays(9, n, k) for k in (1088, 1536, 1600, 2048, 2560, 2624, 3008, 3072, 3136, 4096)] == [True, True, False, False, False, True, True, False, True, True]
    assert [pays(16, 49152, k) for k in (1088, 2048, 3072, 3584)] == [False, False, False, True]
    assert [pays(16, 65536, k) for k in (2048, 3584)] == [False, True] and [pays(16, 151936, k) for k in (3584, 4096)] == [False, True]


def test_where_blocks_with_x_in_registers_stay_better():
    from jax_vllm_amd.ops.kernels import thin_slots as slots

    assert [slots(1, 256, k) for k in (512, 576, 1024, 1088)] == [2] * 4 and [slots(1, n, 1024) for n in (260, 1024, 1028)] == [None, None, 4]
    assert slots(2, 512, 512) == 2 and slots(2, 512, 576) is None and slots(3, 512, 576) == 4
    assert [slots(4, n, 1024) for n in (4096, 4100, 8192, 8196)] == [4, None, None, None] and slots(4, 4100, 1088) == 2
    assert [slots(5, n, 512) for n in (4100, 8192, 8196)] == [2, 2, None]
    assert [slots(9, n, 1024) for n in (4096, 4100, 6144, 6148)] == [4, None, None, 2] and slots(9, 5120, 512) == 2
    assert slots(1, 32000, 2048) == 4 and slots(16, 24576, 4096) == 2


def test_tiles_are_counted_against_the_device_s_units():
    from jax_vllm_amd.ops import kernels

    # 384 tiles: one round of 384 units and no need for two a block, two rounds of 192
    assert [kernels.thin_tiles(16, 6144, cus) for cus in (192, 256, 384)] == [2, 2, 1]
    assert [kernels.thin_tiles_pay(16, 6144, 4096, cus) for cus in (192, 256, 384)] == [True, True, False]
    assert [kernels.thin_slots(16, 24576, 2048, cus) for cus in (256, 1536)] == [2, 4]
    assert kernels._stream_rows_plan(16, torch.empty(6144, 4096, dtype=torch.bfloat16), True, False, None) == "thin"      # planned for, on the CPU


@pytest.mark.gpu
def test_products_ask_for_the_device_s_units(monkeypatch):
    x, w = randn(16, 2048, seed=1).bfloat16(), randn(6144, 2048, seed=2).bfloat16()
    rows = K().StreamRows(x, torch.rand(16, 256, device="cuda") + 0.1, 2048, 1e-6)
    asked, tiles = [], K().thin_tiles
    monkeypatch.setattr(K(), "compute_units", lambda device: 384)
    monkeypatch.setattr(K(), "thin_tiles", lambda m, n, cus=256: asked.append(cus) or tiles(m, n, cus))
    for product in (lambda: K().linear(x, w), lambda: K().gemm_few(x, w, 16), lambda: K().linear(rows, w, gate_pairs="silu")):
        asked.clear()
        product()
        assert asked and set(asked) == {384}
