"""Rows of x that the blocks of a product make themselves: the residual step with its norm, and the splits of a decode attention."""
import math

import pytest
import torch

from .test_kernels_gpu import K, randn

BF = torch.bfloat16


def pending(m, k, n_parts, seed):
    h, w = randn(m, k, seed=seed), 1 + 0.1 * randn(k, seed=seed + 1)
    parts = randn(n_parts, m, k, seed=seed + 2, scale=0.5) if n_parts else None
    return h, parts, w, torch.full_like(h, float("nan"))


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 2])
@pytest.mark.parametrize("n,k,n_parts,gate", [
    (16384 + 32, 1024, 4, True), (20480, 2560, 1, True), (17408, 5120, 3, True),      # blocks that stay, the whole inner size a block
    (6144, 2048, 2, True), (100, 1024, 0, True), (4608, 2048, 4, True), (12288, 4096, 3, True),     # few rows by tiles of 16 and of 32
    (3072, 2048, 4, False), (36, 2048, 0, False), (6144, 4096, 1, False), (2564, 5120, 2, False)])     # the inner size shared out
def test_residual_rows(m, n, k, n_parts, gate):
    k_ = K()
    h, parts, w, out = pending(m, k, n_parts, n)
    W = randn(n, k, dtype=BF, seed=k, scale=k ** -0.5)
    eps, options = 1e-6, dict(gate_pairs="silu") if gate else dict(partial_ok=True, partial_max_width=None)
    assert k_.linear_takes_pending_rows(m, W, gate_pairs=gate, **{} if gate else options)
    got = k_.linear(k_.PendingRows(h, parts, w, eps, out), W, **options)
    v = h.double() + (parts.double().sum(0) if n_parts else 0.0)
    torch.testing.assert_close(out.double(), v, rtol=2e-7 * (n_parts + 1), atol=1e-6)
    assert torch.equal(h, randn(m, k, seed=n))
    x = (v.float() * w).to(BF).double() * torch.rsqrt((v * v).mean(-1, keepdim=True) + eps)      # x is rounded before its scale
    want = x @ W.double().T
    if gate:
        g, u = want[:, 0::2], want[:, 1::2]
        want = torch.nn.functional.silu(g) * u
        assert got.dtype == BF and got.shape == (m, n // 2)
        torch.testing.assert_close(got.double(), want, rtol=2 ** -7, atol=2e-3)                  # bfloat16 results of float sums
    else:
        assert isinstance(got, k_.UnscaledParts) and got.parts.shape[1:] == (m, n)
        sq = got.ssq[:, :got.parts.shape[0]].double().sum(-1, keepdim=True)
        torch.testing.assert_close(sq, (v * v).sum(-1, keepdim=True), rtol=1e-5, atol=0)
        scaled = got.parts.double().sum(0) * torch.rsqrt(sq / got.width + got.eps)
        # a row of x whose float sum lies at a rounding's border may round the other way: a unit of 2^-8 of a few of k terms
        torch.testing.assert_close(scaled, want, rtol=1e-3, atol=2e-3)


@pytest.mark.gpu
@pytest.mark.parametrize("sinks", [False, True])
@pytest.mark.parametrize("m,heads,d,splits,n", [(1, 16, 128, 2, 2048), (2, 16, 128, 8, 2048), (1, 32, 128, 16, 4096), (2, 40, 128, 9, 5120), (1, 64, 64, 5, 1024)])
def test_split_heads(m, heads, d, splits, n, sinks):
    """The merge of the splits and the product behind it; an empty split's rows may hold anything."""
    k_ = K()
    k = heads * d
    W = randn(n, k, dtype=BF, seed=1, scale=k ** -0.5)
    acc, ml = randn(m, heads, splits, d, seed=2), randn(m, heads, splits, 2, seed=3).abs()
    ml[:, ::3, 1] = torch.tensor([float("-inf"), 0.0], device="cuda")
    acc[:, ::3, 1] = float("nan")
    scratch = torch.cat([acc.reshape(-1), ml.reshape(-1)])
    sink = randn(heads, seed=4) if sinks else None
    assert k_.linear_takes_split_heads(m, W, splits) and not k_.linear_takes_split_heads(m, W, 1) and not k_.linear_takes_split_heads(m, W, 17)
    got = k_.linear(k_.SplitHeads(scratch, m, splits, heads, d, sink), W, partial_ok=True)
    top, den = ml[..., 0].double().amax(-1, keepdim=True), ml[..., 1].double()
    f = torch.exp2(ml[..., 0].double() - top)
    num = (torch.where(f[..., None] > 0, acc.double(), 0.0) * f[..., None]).sum(-2)
    den = (den * f).sum(-1)
    if sinks:
        den = den + torch.exp2(sink.double() * math.log2(math.e) - top[..., 0])
    x = (num / den[..., None]).reshape(m, k)
    # x and the two operands' product: a unit of 2^-9 of a row's terms, over k of them
    torch.testing.assert_close(got.double().sum(0), x @ W.double().T, rtol=1e-2, atol=2e-2)
    assert got.shape[1:] == (m, n)


@pytest.mark.gpu
def test_who_may_be_asked():
    k_ = K()
    W = randn(3072, 2048, dtype=BF)
    assert k_.linear_takes_pending_rows(2, W, partial_ok=True) and not k_.linear_takes_pending_rows(3, W, partial_ok=True)
    assert not k_.linear_takes_pending_rows(1, W.float(), partial_ok=True) and not k_.linear_takes_pending_rows(1, W[:, :1999], partial_ok=True)
    h, parts, w, out = pending(1, 2048, 2, 5)
    with pytest.raises(k_.KernelArgumentError, match="from one float tensor"):
        k_.PendingRows(h, parts, w, 1e-6, h)
    with pytest.raises(k_.KernelArgumentError, match="partial products"):
        k_.PendingRows(h, randn(5, 1, 2048), w, 1e-6, out)
    with pytest.raises(k_.KernelArgumentError, match="at most 2 rows"):
        k_.PendingRows(randn(3, 2048), None, w, 1e-6, randn(3, 2048))
    with pytest.raises(k_.KernelArgumentError, match="ask linear_takes"):
        k_.linear(k_.PendingRows(randn(1, 1536), None, randn(1536), 1e-6, randn(1, 1536)), randn(64, 1536, dtype=BF))


@pytest.mark.gpu
@pytest.mark.parametrize("graphs", [True, False])
def test_a_model_of_few_requests_like_one_of_three(graphs):
    """Decoding alone, by two and by three requests (whose rows are made by launches of their own): the same logits within rounding."""
    from jax_vllm_amd import LLM
    from jax_vllm_amd.config.registry import resolve
    from jax_vllm_amd.engine.entries import StepEntry
    from jax_vllm_amd.ops import kernels as kernels_
    from jax_vllm_amd.parts.model import DecoderModel

    cfg = dict(architectures=["Qwen3ForCausalLM"], head_dim=128, rope_theta=1e6, rms_norm_eps=1e-6, tie_word_embeddings=False, max_position_embeddings=4096,
               num_hidden_layers=3, hidden_size=2048, num_attention_heads=16, num_key_value_heads=4, intermediate_size=1024, vocab_size=512)
    arch, typed, _ = resolve(cfg)
    model = DecoderModel(arch.build_spec(typed))
    g = torch.Generator().manual_seed(3)
    tensors = {name: ((1 + 0.05 * torch.randn(t.shape, generator=g)) if len(t.shape) == 1 else torch.randn(t.shape, generator=g) * t.shape[-1] ** -0.5)
               for name, t in model.tensor_specs().items()}
    model.bind({n: t.cuda().to(BF if model.tensor_specs()[n].role == "matrix" else torch.float32) for n, t in tensors.items()}, BF)
    made = []
    linear_made = kernels_._linear_made
    kernels_._linear_made = lambda x, *a: made.append(type(x).__name__) or linear_made(x, *a)
    try:
        def decode(groups):
            llm = LLM(model, dtype="bf16", block_size=16, num_blocks=200, max_num_seqs=4, max_model_len=900, max_num_batched_tokens=2048,
                      use_hip_graphs=graphs, enable_prefix_cache=False)
            prompts = [torch.randint(0, 512, (n,), generator=torch.Generator().manual_seed(n)).tolist() for n in (300, 17, 700)]
            out = [[] for _ in prompts]
            for group in groups:
                for i in group:
                    llm.core.start_request(i)
                llm.core.run([StepEntry(i, prompts[i], []) for i in group])
                for step in range(4):
                    logits = llm.core.run([StepEntry(i, [5 + 7 * step + i], [0]) for i in group])
                    for i, row in zip(group, logits):
                        out[i].append(row.clone())
            return torch.stack([torch.stack(o) for o in out])

        want = decode([(0, 1, 2)])
        assert not made
        for groups in ([(0,), (1,), (2,)], [(0, 2), (1,)]):
            got = decode(groups)
            assert made.count("PendingRows") >= 6 and made.count("SplitHeads") >= 3
            # bfloat16 layers: what two orders of sums differ by, as in the step's own error against float64
            assert ((got - want).norm() / want.norm()).item() < 1.2e-2
            made.clear()
    finally:
        kernels_._linear_made = linear_made


def test_when_the_output_product_merges(monkeypatch):
    """One row up to 8 splits always; more splits, or two rows, while no unit gets a second block (or tile) to read them for."""
    from jax_vllm_amd.ops import kernels

    monkeypatch.setattr(kernels, "compute_units", lambda device: 256)
    pays = lambda m, n, k, splits: kernels.split_heads_pay(m, torch.empty(n, k, dtype=BF), splits)
    shapes = [(2048, 2048), (4096, 4096), (5120, 5120), (2560, 4096), (6144, 2048), (8192, 8192)]
    assert all(pays(1, n, k, splits) for n, k in shapes for splits in (2, 8)) and not any(pays(1, n, k, 1) for n, k in shapes)
    assert [pays(1, n, k, 16) for n, k in shapes] == [True, False, True, False, False, True]
    assert [pays(2, n, k, 8) for n, k in shapes] == [True, False, False, False, False, False]
    assert not any(pays(2, n, k, 16) or pays(1, n, k, 17) or pays(3, n, k, 4) for n, k in shapes)
    assert not pays(1, 8192, 10240, 16) and pays(1, 8192, 10240, 8) and pays(2, 1024, 4096, 4) and not pays(2, 1040, 4096, 4)


@pytest.mark.gpu
@pytest.mark.parametrize("graphs", [True, False])
def test_a_mixer_that_leaves_no_parts(graphs):
    """An output product whose inner size (512) is not shared out leaves bfloat16 rows: the stream goes through the second norm's launch and back
    into its own buffer.  One and two requests as three, whose rows are made by launches of their own."""
    from jax_vllm_amd import LLM
    from jax_vllm_amd.config.registry import resolve
    from jax_vllm_amd.engine.entries import StepEntry
    from jax_vllm_amd.ops import kernels as kernels_
    from jax_vllm_amd.parts.model import DecoderModel

    cfg = dict(architectures=["Qwen3ForCausalLM"], head_dim=128, rope_theta=1e6, rms_norm_eps=1e-6, tie_word_embeddings=False, max_position_embeddings=4096,
               num_hidden_layers=3, hidden_size=2048, num_attention_heads=4, num_key_value_heads=2, intermediate_size=1024, vocab_size=512)
    arch, typed, _ = resolve(cfg)
    model = DecoderModel(arch.build_spec(typed))
    g = torch.Generator().manual_seed(4)
    tensors = {name: ((1 + 0.05 * torch.randn(t.shape, generator=g)) if len(t.shape) == 1 else torch.randn(t.shape, generator=g) * t.shape[-1] ** -0.5)
               for name, t in model.tensor_specs().items()}
    model.bind({n: t.cuda().to(BF if model.tensor_specs()[n].role == "matrix" else torch.float32) for n, t in tensors.items()}, BF)
    made = []
    linear_made = kernels_._linear_made
    kernels_._linear_made = lambda x, *a: made.append(type(x).__name__) or linear_made(x, *a)
    try:
        def decode(groups):
            llm = LLM(model, dtype="bf16", block_size=16, num_blocks=200, max_num_seqs=4, max_model_len=400, max_num_batched_tokens=2048,
                      use_hip_graphs=graphs, enable_prefix_cache=False)
            prompts = [torch.randint(0, 512, (n,), generator=torch.Generator().manual_seed(n)).tolist() for n in (40, 17, 99)]
            out = [[] for _ in prompts]
            for group in groups:
                for i in group:
                    llm.core.start_request(i)
                llm.core.run([StepEntry(i, prompts[i], []) for i in group])
                for step in range(4):
                    for i, row in zip(group, llm.core.run([StepEntry(i, [5 + 7 * step + i], [0]) for i in group])):
                        out[i].append(row.clone())
            return torch.stack([torch.stack(o) for o in out])

        want = decode([(0, 1, 2)])
        assert not made
        for groups in ([(0,), (1,), (2,)], [(0, 2), (1,)]):
            got = decode(groups)
            # one product a layer makes its rows (the other reads what the norm's launch leaves), as often as the launches run on the host
            assert set(made) == {"PendingRows"} and len(made) % 3 == 0
            assert len(made) <= 3 * 4 * len(groups) if not graphs else made
            assert ((got - want).norm() / want.norm()).item() < 1.2e-2      # bfloat16 layers, as above
            made.clear()
    finally:
        kernels_._linear_made = linear_made
