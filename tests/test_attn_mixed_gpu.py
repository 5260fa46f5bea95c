"""Prompts and decoded tokens of a step in one attention launch: the bits of the two launches it stands for, with and without splits, windows and
sinks; which steps take it."""
import pytest
import torch

from .test_kernels_gpu import K


@pytest.mark.gpu
@pytest.mark.parametrize("nq,nkv,d", [(32, 8, 128), (16, 4, 128), (4, 4, 64), (12, 2, 128)])
@pytest.mark.parametrize("decodes,prompts", [([(700, 1)] * 3, [(0, 65)]), ([(5, 1), (1500, 1)] * 20, [(0, 300), (33, 130)]), ([(90, 1)], [(400, 2)])])
@pytest.mark.parametrize("window,sinks", [(0, False), (100, True), (-64, False)])
def test_the_bits_of_two_launches(monkeypatch, nq, nkv, d, decodes, prompts, window, sinks):
    from types import SimpleNamespace

    from jax_vllm_amd.parts import attention_backend
    from jax_vllm_amd.parts.spec import LayerMemory, StepContext

    g = torch.Generator(device="cuda").manual_seed(d + nq)
    reqs = decodes[1:] + prompts + decodes[:1]          # decoded tokens before and behind the prompts
    lens, ctx, page = [n for _, n in reqs], [c for c, _ in reqs], 16
    need = [-(-(c + n) // page) for c, n in reqs]
    pages = 1 + sum(need)
    order = (torch.randperm(pages - 1, generator=torch.Generator().manual_seed(1)) + 1).tolist()
    tables = torch.zeros(len(reqs), max(need), dtype=torch.int32)
    for r, n in enumerate(need):
        tables[r, :n] = torch.tensor([order.pop() for _ in range(n)])
    k, v = (torch.randn(pages, nkv, page, d, generator=g, device="cuda").bfloat16() for _ in range(2))
    v = v.transpose(2, 3).contiguous()
    n = sum(lens)
    q = torch.randn(n, nq * d, generator=g, device="cuda").bfloat16()

    def i32(values):
        return torch.tensor(values, dtype=torch.int32, device="cuda")

    att = SimpleNamespace(nq=nq, nkv=nkv, d=d, window=window if window > 0 else None, chunk=-window if window < 0 else None, q_row_stride=nq * d,
                          sinks=torch.randn(nq, generator=g, device="cuda") if sinks else None, scale=d ** -0.5)
    taken = []
    mixed = K().attn_mixed
    monkeypatch.setattr(K(), "attn_mixed", lambda *a, **kw: taken.append(1) or mixed(*a, **kw))

    def attention():
        step = StepContext(num_tokens=n, num_requests=len(reqs), positions=i32([c + i for c, m in reqs for i in range(m)]),
                           token_req=i32([r for r, m in enumerate(lens) for _ in range(m)]), cu_seqlens=i32([0] + torch.tensor(lens).cumsum(0).tolist()),
                           context_lens=i32(ctx), slot_ids=i32([0] * len(reqs)), block_tables=[tables.cuda()], slot_mappings=[None], page_size=page,
                           q_lens_host=lens, context_lens_host=ctx, slot_ids_host=[0] * len(reqs), max_q_len=max(lens), max_kv_len=max(c + m for c, m in reqs))
        out = torch.full((n, nq * d), float("nan"), dtype=torch.bfloat16, device="cuda")
        attention_backend.run(att, out, q, step, LayerMemory(pages={"k": k, "v": v}, group=0))
        return out

    got = attention()
    assert taken and torch.isfinite(got).all()
    monkeypatch.setattr(K(), "attn_mixed_possible", lambda *a: False)
    assert torch.equal(attention(), got) and len(taken) == 1


@pytest.mark.gpu
def test_which_sizes_take_one_launch():
    fits = K().attn_mixed_possible
    assert fits(128, 16, 512, 32, 8) and fits(64, 16, 512, 16, 16)
    assert not fits(128, 16, 512, 32, 4) and not fits(128, 32, 512, 32, 8) and not fits(256, 16, 512, 16, 1) and not fits(96, 16, 64, 8, 8)
    assert not fits(128, 16, 5000, 32, 8) and not fits(128, 16, 4096, 32, 8)       # a second block would not fit a unit
