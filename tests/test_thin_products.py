"""Products of up to 16 rows through rings of W and x: the residual stream as their result and rows whose scale is still to be applied, against float64;
the bits of blocks with x in registers; a model's layers through the stream against the same layers without."""
import pytest
import torch

from .test_kernels_gpu import K, randn


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 7, 8, 9, 16])
@pytest.mark.parametrize("n,k", [(64, 64), (192, 448), (1088, 576), (2048, 3072), (4096, 4160)])
def test_into_the_stream(m, n, k):
    x, w, h = randn(m, k, seed=m).bfloat16(), randn(n, k, seed=n + k).bfloat16(), randn(m, n, seed=3)
    weight = randn(n, seed=4)
    want = h.double() + x.double() @ w.double().T
    got = h.clone()
    rows = K().gemm_into_stream(got, x, w, weight, 1e-6)
    # exact products, eight chains of k / 8 terms, eight sums and the stream in float
    bound = 2.0 ** -24 * (k / 8 + 9) * (h.double().abs() + x.double().abs() @ w.double().abs().T)
    assert ((got.double() - want).abs() <= bound).all()
    assert torch.equal(rows.x, (got * weight).bfloat16())
    # squares and their sums in float: 16 columns a share
    shares = got.double().square().view(m, n // 16, 16).sum(2)
    assert ((rows.ssq[:, :n // 16].double() - shares).abs() <= 2.0 ** -24 * 17 * shares).all()
    alone = h.clone()
    assert K().gemm_into_stream(alone, x, w) is None and torch.equal(alone, got)
    part = h[m // 2:].clone()
    K().gemm_into_stream(part, x[m // 2:].contiguous(), w)
    assert torch.equal(part, got[m // 2:])      # whatever the batch


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 8, 13])
@pytest.mark.parametrize("n,k,pairs", [(48, 64, True), (3072, 2048, False), (6144, 2048, True), (6144, 4096, False), (24576, 4096, True), (100, 1024, False),
                                       (5120, 1088, False)])
def test_rows_with_many_shares_of_their_scale(m, n, k, pairs):
    h, w = randn(m, k, seed=m) * 3, randn(n, k, seed=n + k).bfloat16()
    weight = 1 + 0.1 * randn(k, seed=5)
    x = (h * weight).bfloat16()
    ssq = torch.full((m, 256), float("nan"), device="cuda")
    ssq[:, :k // 16] = h.square().view(m, k // 16, 16).sum(2)
    rows = K().StreamRows(x, ssq, k, 1e-6)
    assert K().linear_takes_stream_rows(m, w, gate_pairs=pairs, partial_ok=not pairs, partial_max_width=None)
    y = K().linear(rows, w, gate_pairs="silu" if pairs else None, partial_ok=not pairs, partial_max_width=None)
    scale = torch.rsqrt(h.double().square().mean(1, keepdim=True) + 1e-6)
    z = x.double() @ w.double().T * scale
    if pairs:
        g, u = z[:, 0::2], z[:, 1::2]
        torch.testing.assert_close(y.double(), g / (1 + torch.exp(-g)) * u, rtol=2.0 ** -7, atol=1e-3)      # a rounding of bfloat16
        return
    # the product's bound, and the scale's: 256 squares and sums, a root
    bound = 2.0 ** -24 * (k / 8 + 8 + k / 2 + 8) * (x.double().abs() @ w.double().abs().T) * scale
    assert ((y.sum(0).double() - z).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(5, 2048, 1024), (16, 512, 512), (9, 20, 448)])
def test_the_bits_of_blocks_with_x_in_registers(monkeypatch, m, n, k):
    x, w = randn(m, k, seed=m).bfloat16(), randn(n, k, seed=n + k).bfloat16()
    y = K().gemm_few(x, w, 16, out_dtype=torch.float32)
    monkeypatch.setattr(K(), "thin_slots", lambda *_: None)
    assert torch.equal(K().gemm_few(x, w, 16, out_dtype=torch.float32), y) and torch.equal(K().gemm_few(x, w, 32, out_dtype=torch.float32), y)


def test_where_the_stream_takes_a_product():
    from jax_vllm_amd.ops import kernels

    def w(n, k, dtype=torch.bfloat16):
        return torch.empty(n, k, dtype=dtype)

    assert kernels.stream_product_possible(16, w(4096, 64)) and not kernels.stream_product_possible(17, w(4096, 64))
    assert not kernels.stream_product_possible(1, w(4160, 64)) and not kernels.stream_product_possible(1, w(96, 64))
    assert not kernels.stream_product_possible(1, w(64, 96)) and not kernels.stream_product_possible(1, w(64, 64, torch.float32))
    assert not kernels.stream_product_possible(1, w(64, 65)[:, 1:])      # off 16 bytes, and no whole rows


def test_where_a_layer_leaves_its_products_to_the_stream():
    from types import SimpleNamespace

    from jax_vllm_amd.ops.kernels import stream_product_pays as pays
    from jax_vllm_amd.parts.attention import GroupedQueryAttention
    from jax_vllm_amd.parts.mlp import GatedMLP

    assert pays(16, 2048, 8192) and not pays(16, 2048, 8256) and pays(8, 2048, 14336) and not pays(8, 2048, 14400) and not pays(9, 1536, 8960)
    assert pays(1, 1024, 8192) and not pays(1, 1024, 8256) and not pays(16, 512, 12288)
    assert pays(1, 4096, 20480) and not pays(8, 2112, 20544) and pays(9, 2112, 20544) and pays(16, 4096, 12288)

    def w(n, k):
        return torch.empty(n, k, dtype=torch.bfloat16, device="meta")

    class Weight(torch.Tensor):      # (a meta tensor has no address)
        data_ptr = lambda self: 0

    for k, leaves in ((8192, True), (10240, False)):
        weight = w(1024, k).as_subclass(Weight)
        assert GatedMLP.leaves_product(SimpleNamespace(partial_out=True, w_down=weight), 4) == leaves
        assert GroupedQueryAttention.leaves_product(SimpleNamespace(wide=False, filtered=False, b_o=None, w_o=weight), 4) == leaves


@pytest.mark.gpu
@pytest.mark.parametrize("running,prompt", [(1, 0), (3, 0), (16, 0), (0, 12), (2, 9)])
def test_layers_through_the_stream(monkeypatch, running, prompt):
    """Steps of few rows, decoding and prompt tokens, replayed and not: the same logits as with float parts and norms between."""
    from jax_vllm_amd import LLM, write_random_model
    from jax_vllm_amd.engine.entries import StepEntry
    from jax_vllm_amd.parts.block import PreNormBlock
    import tempfile

    config = dict(architectures=["Qwen3ForCausalLM"], num_hidden_layers=3, hidden_size=512, num_attention_heads=4, num_key_value_heads=2, head_dim=128,
                  intermediate_size=768, vocab_size=512, rope_theta=1e4, rms_norm_eps=1e-6, tie_word_embeddings=False, max_position_embeddings=4096)
    through, layers = PreNormBlock._through_stream, config["num_hidden_layers"]
    calls = {"into": 0, "scaled": 0, "through": 0}
    for name, counted in (("gemm_into_stream", "into"), ("gemm_thin_scaled", "scaled")):
        launch = getattr(K(), name)
        monkeypatch.setattr(K(), name, lambda *a, launch=launch, counted=counted: calls.update({counted: calls[counted] + 1}) or launch(*a))

    def asked(self, n, *a):
        ok = through(self, n, *a)
        calls["through"] += ok
        return ok

    def logits_of(folder, on):
        monkeypatch.setattr(PreNormBlock, "_through_stream", asked if on else lambda self, n, *a: False)
        calls.update(into=0, scaled=0, through=0)
        llm = LLM(folder, dtype="bf16", block_size=16, num_blocks=200, max_num_seqs=20, max_model_len=256, max_num_batched_tokens=512, enable_prefix_cache=False)
        for i in range(running):
            llm.core.start_request(i)
            llm.core.run([StepEntry(i, [(7 * i + j) % 512 for j in range(20 + 5 * i)], [])])
        out = []
        for step in range(4):
            entries = [StepEntry(i, [(i + step) % 512], [0]) for i in range(running)]
            if prompt:
                llm.core.start_request(("p", step))
                entries.append(StepEntry(("p", step), [(3 * j + step) % 512 for j in range(prompt)], [0, prompt - 1]))
            out.append(llm.core.run(entries).clone())
        return torch.stack(out)

    with tempfile.TemporaryDirectory() as tmp:
        folder = write_random_model(tmp, config, seed=1, std=0.04, norm_std=0.1)
        a = logits_of(folder, True)
        steps, left = divmod(calls["through"], layers)      # steps that were launched, not replayed
        # every product of a layer joins the stream, all products behind the first norm read it
        assert steps and not left and calls["into"] == steps * 2 * layers and calls["scaled"] == steps * (2 * layers - 1)
        b = logits_of(folder, False)
        assert not any(calls.values())
    # two roundings of bfloat16 a layer and product that differ by the order of sums
    assert ((a - b).norm() / b.norm()).item() < 6 * 2.0 ** -8


def test_where_one_whole_product_stands_for_parts():
    from jax_vllm_amd.ops.kernels import thin_whole_pays as pays

    assert pays(8, 2052, 2048) and not pays(9, 2052, 2048) and not pays(8, 2052, 1984) and not pays(8, 2052, 4160)
    assert pays(1, 4096, 4096) and not pays(1, 4100, 4096) and not pays(1, 2044, 3072)
    assert [pays(8, 2048, k) for k in (2048, 2560, 2624, 3072, 4032, 4096)] == [False, False, True, True, True, False]


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,whole", [(8, 4096, 3072, True), (1, 2052, 2048, True), (8, 2048, 2624, True), (8, 2048, 2560, False), (9, 4096, 3072, False), (8, 4100, 2048, False)])
def test_one_whole_product_and_its_readers(m, n, k, whole):
    """What ``linear`` leaves around the rule, and the launches that add partial products behind it."""
    x, w, h = randn(m, k, seed=m).bfloat16(), randn(n, k, seed=n + k).bfloat16(), randn(m, n, seed=7)
    weight = 1 + 0.1 * randn(n, seed=8)
    parts = K().linear(x, w, partial_ok=True)
    assert (parts.dim() == 3 and parts.shape[0] == 1) == whole
    z = x.double() @ w.double().T
    sums = parts.sum(0) if parts.dim() == 3 else parts
    assert ((sums.double() - z).abs() <= 2.0 ** -24 * k * (x.double().abs() @ w.double().abs().T)).all()      # a sum of k products in float in any order
    if not whole:
        return
    stream, out = h.clone(), torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
    K().add_rmsnorm(stream, parts, weight, out, 1e-6)
    assert torch.equal(stream, h + parts[0])
    want = stream.double() * torch.rsqrt(stream.double().square().mean(1, keepdim=True) + 1e-6) * weight.double()
    torch.testing.assert_close(out.double(), want, rtol=2.0 ** -8, atol=1e-6)
    if n % 512 == 0:
        again = h.clone()
        rows = K().add_parts_unscaled(again, parts, weight, 1e-6)
        assert torch.equal(again, stream) and torch.equal(rows.x, (stream * weight).bfloat16())
