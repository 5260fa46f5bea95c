"""Prefill attention at head size 256 in its two forms (16 and 32 rows a wave): the rule between them, and both against float64."""
import math

import pytest
import torch

from jax_vllm_amd.parts.attention_backend import few_rows_of_256

from .test_f32_path import reference, run_step
from .test_kernels_gpu import K, _mfma_inputs, _mfma_reference, _prefill_work, build_paged


def test_the_rule_of_pages_other_than_16():
    assert few_rows_of_256(300 * 16, 64, 256) and few_rows_of_256(320 * 64, 64, 256) and not few_rows_of_256(320 * 64 + 1, 64, 256)
    assert few_rows_of_256(320 * 64 + 1, 64, 304)


def test_which_rule_a_plan_asks(monkeypatch):
    """Pages of 16 keys: the rule of the halves, which knows the walk; others count rows alone."""
    from types import SimpleNamespace

    from jax_vllm_amd.ops import kernels
    from jax_vllm_amd.parts import attention_backend

    monkeypatch.setattr(kernels, "compute_units", lambda device: 256)
    monkeypatch.setattr(attention_backend, "upload_i32", lambda values, device: torch.tensor(values, dtype=torch.int32))

    def one_group(page_size, tokens, context, window=0):
        ctx = SimpleNamespace(q_lens_host=[tokens], context_lens_host=[context], page_size=page_size, block_tables=[torch.zeros(1, 64)])
        return attention_backend.plan_mfma(ctx, 16, 1, 256, window, "cpu").one_group

    assert one_group(16, 300, 0) is False and one_group(16, 250, 0) and one_group(16, 300, 100000) is False
    for page_size in (8, 24, 32, 64):
        assert one_group(page_size, 300, 0) and one_group(page_size, 1280, 100000) and not one_group(page_size, 1281, 0, 128)


@pytest.mark.gpu
@pytest.mark.parametrize("plan", ["single", "planner", "far", "one_group"])
@pytest.mark.parametrize("case", [
    # nq, nkv, page_size, (context, tokens), window
    (4, 2, 16, [(0, 1), (0, 64), (5, 131)], None),
    (16, 1, 16, [(0, 70), (300, 9)], 100),
    (6, 2, 8, [(0, 65), (63, 33)], None),           # 3 heads a group, pages of 8
    (4, 1, 64, [(130, 100)], 64),
    (4, 4, 24, [(0, 77), (40, 64)], None),          # pages that are no power of two
    (2, 1, 128, [(200, 130)], None),                # pages larger than a key tile
    (8, 1, 16, [(1900, 40)], 1024),
])
def test_both_forms(case, plan):
    nq, nkv, page_size, reqs, window = case
    d, one = 256, plan == "one_group"
    qs, ks, vs, dev = _mfma_inputs(nq, nkv, d, page_size, reqs)
    work, n_work = _prefill_work(reqs, nq // nkv, d, window, "single" if one else plan)
    out = torch.full((dev["n"], nq * d), float("nan"), dtype=torch.bfloat16).cuda()
    K().attn_prefill_mfma(out, dev["q"], dev["stride"], dev["k_pages"], dev["v_pages"], dev["tables"], dev["cu"], dev["ctx"],
                          work, n_work, nq, nkv, d, 1.0 / math.sqrt(d), window or 0, one_group=one)
    ref = _mfma_reference(qs, ks, vs, reqs, 1.0 / math.sqrt(d), window, nq, d)
    torch.testing.assert_close(out.double().cpu(), ref, rtol=2e-2, atol=2e-2)       # probabilities and results in 8 bits of fraction


@pytest.mark.gpu
@pytest.mark.parametrize("d", [32, 64, 128, 256])
@pytest.mark.parametrize("tokens", [16, 40])                # items whose second pair of waves, and second wave, have no rows
def test_the_first_keys_of_a_walk_of_three_tiles_and_more(d, tokens):
    """Pages of 16: the third tile's keys are loaded where the first tile's were, which every wave must have read by then,
    also beside waves that have no rows and do not read.  Warm keys arrive soonest, so each launch is repeated."""
    nq, nkv, page_size = 4, 2, 16
    reqs = [(112, tokens), (300, tokens), (0, 200)]         # three tiles exactly, several, and growing walks
    qs, ks, vs, dev = _mfma_inputs(nq, nkv, d, page_size, reqs)
    work, n_work = _prefill_work(reqs, nq // nkv, d, None, "single")
    ref = _mfma_reference(qs, ks, vs, reqs, 1.0 / math.sqrt(d), None, nq, d)
    first = None
    for _ in range(5):
        out = torch.full((dev["n"], nq * d), float("nan"), dtype=torch.bfloat16).cuda()
        K().attn_prefill_mfma(out, dev["q"], dev["stride"], dev["k_pages"], dev["v_pages"], dev["tables"], dev["cu"], dev["ctx"],
                              work, n_work, nq, nkv, d, 1.0 / math.sqrt(d))
        torch.testing.assert_close(out.double().cpu(), ref, rtol=2e-2, atol=2e-2)   # probabilities and results in 8 bits of fraction
        first = out if first is None else first
        assert torch.equal(out, first)


MASKS = [{"window": 100}, {"window": 100, "keep": 20}, {"window": 70, "keep": 200}, {"chunk": 96}, {"chunk": 64, "keep": 33}, {}]


@pytest.mark.gpu
@pytest.mark.parametrize("page_size", [16, 24, 64])
@pytest.mark.parametrize("one_group", [True, False])
@pytest.mark.parametrize("mask", MASKS, ids=str)
def test_both_forms_with_sinks_caps_kept_keys_and_blocks(mask, one_group, page_size):
    nq, nkv, d, scale = 6, 2, 256, 0.09
    reqs = [(0, 70), (230, 90), (5, 131)]
    qs, ks, vs, dev = _mfma_inputs(nq, nkv, d, page_size, reqs)
    sinks = torch.linspace(-1.0, 2.0, nq)
    window, chunk, keep = mask.get("window"), mask.get("chunk"), mask.get("keep", 0)
    for cap, with_sinks in ((0.0, True), (3.0, False), (3.0, True)):
        work, n_work = _prefill_work(reqs, nq // nkv, d, window, "single" if one_group else "neighbours")
        out = torch.full((dev["n"], nq * d), float("nan"), dtype=torch.bfloat16).cuda()
        K().attn_prefill_mfma(out, dev["q"], dev["stride"], dev["k_pages"], dev["v_pages"], dev["tables"], dev["cu"], dev["ctx"], work, n_work,
                              nq, nkv, d, scale, K().key_window(window, chunk), sinks=sinks.cuda() if with_sinks else None, cap=cap, keep=keep,
                              one_group=one_group)
        want = torch.cat([reference(q, k, v, torch.arange(c, c + n), scale, window, chunk, keep, cap, sinks if with_sinks else None)
                          for q, k, v, (c, n) in zip(qs, ks, vs, reqs)]).reshape(-1, nq * d)
        torch.testing.assert_close(out.double().cpu(), want, rtol=2e-2, atol=2e-2)      # probabilities and results in 8 bits of fraction


@pytest.mark.gpu
@pytest.mark.parametrize("reqs,page_size,mask,one_group", [
    ([(0, 70), (300, 9), (40, 1)], 16, {"window": 100, "keep": 20}, True),              # few rows
    ([(0, 1400), (40, 1)], 16, {"window": 300, "keep": 20}, False),                     # more than 320 groups
    ([(0, 1400)], 16, {"chunk": 256}, True),                                            # short walks
    ([(2100, 30)], 16, {}, False),                                                      # many keys
    ([(2100, 30)], 32, {}, True),                                                       # but pages of 32
    ([(0, 1400)], 32, {"chunk": 256, "keep": 5}, False),
])
def test_the_plan_and_its_kernel(reqs, page_size, mask, one_group):
    """The backend's plan at head size 256 on each side of the rule: its items and the form it names belong together (an item of
    two groups in the form of one would leave half its rows out)."""
    nq, nkv, d = 16, 1, 256
    g = torch.Generator().manual_seed(7)
    bf = torch.bfloat16
    ks, vs = ([torch.randn(c + n, nkv, d, generator=g).to(bf).float() for c, n in reqs] for _ in range(2))
    qs = [torch.randn(n, nq, d, generator=g).to(bf).float() for _, n in reqs]
    *pages, tables = build_paged(ks, vs, page_size)
    sinks, plans = torch.linspace(-1.0, 2.0, nq), []
    out = run_step((nq, nkv, d, page_size), reqs, pages, tables, qs, **mask, cap=4.0, sinks=sinks.cuda(), dtype=bf, plans=plans)
    plan, = plans
    assert plan.one_group == one_group
    assert bool((plan.prefill_work.view(-1, 3)[:, 2] >= 0).any()) == (not one_group)
    want = torch.cat([reference(q, k, v, torch.arange(c, c + n), d ** -0.5, mask.get("window"), mask.get("chunk"), mask.get("keep", 0), 4.0, sinks)
                      for q, k, v, (c, n) in zip(qs, ks, vs, reqs)]).reshape(-1, nq * d)
    torch.testing.assert_close(out.double(), want, rtol=2e-2, atol=2e-2)
