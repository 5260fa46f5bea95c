"""32-bit products of up to 8 rows that join the residual stream in their own launch, and those that apply the rows' scale."""
import pytest
import torch

from .test_kernels_gpu import K, randn


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 5, 8])
@pytest.mark.parametrize("n,k", [(4, 4), (36, 100), (2048, 3072), (2052, 64), (4096, 36)])
def test_into_the_stream(m, n, k):
    h, x, w, weight = randn(m, n, seed=1), randn(m, k, seed=2), randn(n, k, seed=3), randn(n, seed=4)
    want = h + K().gemm_f32(x, w)
    got, alone = h.clone(), h.clone()
    rows = K().gemm_into_stream(got, x, w, weight, 1e-6)
    assert torch.equal(got, want) and torch.equal(rows.x, want * weight)
    share = -(-n // rows.shares)
    sums = torch.nn.functional.pad(want.double() ** 2, (0, share * rows.shares - n)).view(m, rows.shares, share).sum(-1)
    assert share in (8, 16) or rows.shares == 1
    torch.testing.assert_close(rows.ssq[:, :rows.shares].double(), sums, rtol=16 * 2.0 ** -24, atol=0)      # 15 additions of positive numbers
    assert K().gemm_into_stream(alone, x, w) is None and torch.equal(alone, want)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 5, 8])
@pytest.mark.parametrize("n,k,shares", [(8, 36, 3), (2048, 4096, 256), (3072, 2048, 256), (3074, 100, 13), (6144, 2048, 128), (6146, 2052, 171)])
@pytest.mark.parametrize("pairs", [False, True])
def test_scaled_rows(m, n, k, shares, pairs):
    x, w = randn(m, k, seed=5), randn(n, k, seed=6)
    ssq = torch.full((m, 256), float("nan"), device="cuda")                    # shares that nobody wrote are not read
    ssq[:, :shares] = randn(m, shares, seed=7) ** 2
    rows = K().StreamRows(x, ssq, k, 1e-6, -(-k // shares))
    assert rows.shares == shares and K().linear_takes_stream_rows(m, w, gate_pairs=pairs)
    scale = (ssq[:, :shares].double().sum(-1, keepdim=True) / k + 1e-6).rsqrt()
    want = K().gemm_f32(x, w).double() * scale
    if pairs:
        want = torch.nn.functional.silu(want[:, 0::2]) * want[:, 1::2]
    got = K().linear(rows, w, gate_pairs="silu" if pairs else None)
    # the scale's sum of 256, its root and one rounding of the product; the activation's exponential and two more
    torch.testing.assert_close(got.double(), want, rtol=(300 if pairs else 20) * 2.0 ** -24, atol=1e-6 * float(want.abs().max()))


def test_which_products_join_the_stream():
    from jax_vllm_amd.ops import kernels

    def w(n, k):
        return torch.empty(n, k)

    assert kernels.f32_stream_product_possible(8, w(4096, 4)) and not kernels.f32_stream_product_possible(9, w(64, 64))
    assert not kernels.f32_stream_product_possible(1, w(4100, 8)) and not kernels.f32_stream_product_possible(1, w(6, 8))
    assert not kernels.f32_stream_product_possible(1, w(8, 6)) and not kernels.f32_stream_product_possible(1, torch.empty(8, 8, dtype=torch.bfloat16))
    assert not kernels.linear_takes_stream_rows(9, w(64, 64)) and not kernels.linear_takes_stream_rows(1, w(64, 5000))
    assert kernels.linear_takes_stream_rows(8, w(6144, 2048), gate_pairs=True)


@pytest.mark.gpu
@pytest.mark.parametrize("running,prompt", [(1, 0), (5, 0), (0, 8), (2, 5)])
def test_layers_through_the_stream(monkeypatch, running, prompt):
    """Steps of few rows, replayed and not: the logits of norms between the products."""
    from jax_vllm_amd import LLM, write_random_model
    from jax_vllm_amd.engine.entries import StepEntry
    from jax_vllm_amd.parts.block import PreNormBlock
    import tempfile

    config = dict(architectures=["Qwen3ForCausalLM"], num_hidden_layers=3, hidden_size=328, num_attention_heads=4, num_key_value_heads=2, head_dim=64,
                  intermediate_size=500, vocab_size=300, rope_theta=1e4, rms_norm_eps=1e-6, tie_word_embeddings=False, max_position_embeddings=4096)
    used = []
    through = PreNormBlock._through_stream

    def logits_of(folder, on):
        def choose(self, n, *parts):
            used.append(on and through(self, n, *parts))
            return used[-1]

        monkeypatch.setattr(PreNormBlock, "_through_stream", choose)
        llm = LLM(folder, dtype="fp32", block_size=16, num_blocks=200, max_num_seqs=20, max_model_len=256, max_num_batched_tokens=512, enable_prefix_cache=False)
        for i in range(running):
            llm.core.start_request(i)
            llm.core.run([StepEntry(i, [(7 * i + j) % 300 for j in range(20 + 5 * i)], [])])
        out = []
        for step in range(4):
            entries = [StepEntry(i, [(i + step) % 300], [0]) for i in range(running)]
            if prompt:
                llm.core.start_request(("p", step))
                entries.append(StepEntry(("p", step), [(3 * j + step) % 300 for j in range(prompt)], [0, prompt - 1]))
            out.append(llm.core.run(entries).clone())
        return torch.stack(out)

    with tempfile.TemporaryDirectory() as tmp:
        folder = write_random_model(tmp, config, seed=1, std=0.04, norm_std=0.1)
        a, b = logits_of(folder, True), logits_of(folder, False)
    assert any(used)
    # a few roundings of 32 bits a layer
    assert ((a - b).norm() / b.norm()).item() < 40 * 2.0 ** -24
