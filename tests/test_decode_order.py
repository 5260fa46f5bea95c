"""The order in which a decode attention's blocks take their requests: the device's ranking against the host's, and the same results in any order."""
import math

import pytest
import torch

from .test_kernels_gpu import K, randn


def places(n, at_once):
    """The rank (0: the longest) of the request at each place: the units that get a second request begin with the shorter of the first lap.
    What the device's order is compared with; the two tests below look at this rule and at the order that the device makes."""
    second = n - at_once
    if second <= 0:
        return list(range(n))
    if n <= 2 * at_once:
        return list(range(at_once - second, at_once)) + list(range(at_once - second)) + list(range(n - 1, at_once - 1, -1))
    order = []
    for lap, first in enumerate(range(0, n, at_once)):
        ranks = list(range(first, min(n, first + at_once)))
        order += ranks[::-1] if lap & 1 else ranks
    return order


@pytest.mark.parametrize("n,at_once", [(33, 32), (40, 32), (63, 32), (64, 32), (5, 3)])
def test_two_a_unit_share_evenly(n, at_once):
    order = places(n, at_once)
    assert sorted(order) == list(range(n))
    sums = {order[j] + order[j + at_once] for j in range(n - at_once)}
    assert len(sums) == 1 and sorted(order[n - at_once:at_once]) == list(range(2 * at_once - n))      # who is alone is among the longest


@pytest.mark.gpu
@pytest.mark.parametrize("n,at_once", [(33, 32), (40, 32), (63, 32), (64, 32), (200, 128), (5, 3)])
def test_two_a_unit_share_evenly_on_the_device(n, at_once):
    """Lengths one apart: every unit with two requests has the same number of keys in all, and who is alone is among the longest."""
    lens = torch.randperm(n, generator=torch.Generator().manual_seed(n)).to(torch.int32)
    order = K().decode_order(lens.cuda(), at_once).tolist()
    seen = [int(lens[i]) for i in order]
    assert sorted(order) == list(range(n)) and len({seen[j] + seen[j + at_once] for j in range(n - at_once)}) == 1
    assert all(v >= n - at_once for v in seen[n - at_once:at_once])


@pytest.mark.gpu
@pytest.mark.parametrize("window", [0, 300, -128])
@pytest.mark.parametrize("n,at_once", [(1, 1), (2, 1), (31, 32), (33, 32), (40, 32), (64, 32), (97, 32), (257, 64), (1024, 256), (1022, 7)])
def test_order_on_the_device(n, at_once, window):
    lens = torch.randint(0, 700 if n < 64 else 90, (n,), generator=torch.Generator().manual_seed(n), dtype=torch.int32)      # equal ones among them
    seen = [min(v, window) if window > 0 else v % -window if window < 0 else v for v in lens.tolist()]
    ranked = sorted(range(n), key=lambda i: (-seen[i], i))
    assert K().decode_order(lens.cuda(), at_once, window).tolist() == [ranked[q] for q in places(n, at_once)]


@pytest.mark.gpu
def test_results_do_not_depend_on_it():
    k_, n, nq, nkv, d, page = K(), 35, 16, 8, 128, 16
    lens = [(37 * i) % 601 for i in range(n)]
    pages = [c // page + 1 for c in lens]
    tables = torch.zeros(n, max(pages), dtype=torch.int32)
    at = 1
    for i, m in enumerate(pages):
        tables[i, :m] = torch.arange(at, at + m)
        at += m
    slots = torch.tensor([int(tables[i, c // page]) * page + c % page for i, c in enumerate(lens)], dtype=torch.int32).cuda()
    kp, vp = randn(at, nkv, page, d, dtype=torch.bfloat16, seed=1), randn(at, nkv, d, page, dtype=torch.bfloat16, seed=2)
    qkv, tables, ctx = randn(n, (nq + 2 * nkv) * d, dtype=torch.bfloat16, seed=3), tables.cuda(), torch.tensor(lens, dtype=torch.int32).cuda()
    cu = torch.arange(n + 1, dtype=torch.int32).cuda()
    order, results = k_.decode_order(ctx, 32), []
    for work in (None, order, order.flip(0).contiguous()):
        k, v, out = kp.clone(), vp.clone(), torch.zeros(n, nq * d, dtype=torch.bfloat16, device="cuda")
        k_.attn_decode_token(out, qkv, slots, None, None, 0.0, None, 0, k, v, tables, ctx, nq, nkv, d, 1 / math.sqrt(d), work=work)
        ready = torch.zeros_like(out)
        k_.attn_decode_mfma(ready, qkv, (nq + 2 * nkv) * d, k, v, tables, cu, ctx, work, n, nq, nkv, d, 1 / math.sqrt(d))
        results.append((out, ready, k, v))
    for other in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(results[0], other))
    with pytest.raises(k_.KernelArgumentError):
        k_.decode_order(torch.zeros(1025, dtype=torch.int32, device="cuda"), 32)


@pytest.mark.gpu
def test_steps_of_a_model_take_their_order_each_time(monkeypatch):
    """Steps of more requests than go to the units at once, eager and replayed: the order is made on the device in every step, also a replayed one whose
    requests have changed places, and the logits are those without an order."""
    from jax_vllm_amd import LLM
    from jax_vllm_amd.config.registry import resolve
    from jax_vllm_amd.engine.entries import StepEntry
    from jax_vllm_amd.parts import attention_backend
    from jax_vllm_amd.parts.model import DecoderModel

    cfg = dict(architectures=["Qwen3ForCausalLM"], head_dim=128, rope_theta=1e6, rms_norm_eps=1e-6, tie_word_embeddings=False, max_position_embeddings=4096,
               num_hidden_layers=2, hidden_size=512, num_attention_heads=8, num_key_value_heads=8, intermediate_size=512, vocab_size=256)
    arch, typed, _ = resolve(cfg)
    model = DecoderModel(arch.build_spec(typed))
    g = torch.Generator().manual_seed(3)
    tensors = {name: ((1 + 0.05 * torch.randn(t.shape, generator=g)) if len(t.shape) == 1 else torch.randn(t.shape, generator=g) * t.shape[-1] ** -0.5)
               for name, t in model.tensor_specs().items()}
    model.bind({n: t.cuda().to(torch.bfloat16 if model.tensor_specs()[n].role == "matrix" else torch.float32) for n, t in tensors.items()}, torch.bfloat16)
    n, at_once = 36, 32
    lengths = [[40 + (37 * i) % 500 for i in range(n)], [530 - (53 * i) % 450 for i in range(n)]]      # a second set of requests in the same rows
    plain, made = attention_backend._decode_work, []

    def with_order(ctx, plan, att, window):
        work = plain(ctx, plan, att, window)
        if work is not None:
            made.append(work)
        return work

    def steps(graphs, choose):
        monkeypatch.setattr(attention_backend, "_decode_work", choose)
        llm = LLM(model, dtype="bf16", block_size=16, num_blocks=2000, max_num_seqs=40, max_model_len=600, max_num_batched_tokens=4096,
                  use_hip_graphs=graphs, enable_prefix_cache=False)
        out = []
        for turn, lens in enumerate(lengths):
            for i, length in enumerate(lens):
                llm.core.start_request((turn, i))
                llm.core.run([StepEntry((turn, i), [(7 * i + j) % 256 for j in range(length)], [])])
            for step in range(3):
                replays = llm.core.graph_replays
                out.append(llm.core.run([StepEntry((turn, i), [(5 + 7 * step + i) % 256], [0]) for i in range(n)]).clone())
                if choose is with_order and (not graphs or llm.core.graph_replays > replays):      # (a step that records runs beside its recording)
                    order = made[-1].tolist()                           # replayed: what the recording's launch has left
                    now = [length + step for length in lens] + [0] * (len(order) - n)      # rows that fill a recorded step up have no keys
                    ranked = sorted(range(len(order)), key=lambda i: (-now[i], i))
                    assert order == [ranked[p] for p in places(len(order), at_once)]
            for i in range(n):
                llm.core.finish_request((turn, i))
        assert not graphs or llm.core.graph_replays >= 5
        return torch.stack(out)

    want = steps(False, lambda ctx, plan, att, window: plan.decode_work)
    for graphs in (False, True):
        made.clear()
        got = steps(graphs, with_order)
        assert made
        if graphs:      # rows that fill the step up: products of another size, bfloat16 layers
            assert ((got - want).norm() / want.norm()).item() < 1.2e-2
        else:
            assert torch.equal(got, want)
