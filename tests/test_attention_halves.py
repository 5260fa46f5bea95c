"""Prefill attention at head size 256 and pages of 16, two waves to 32 rows: walks of one tile to several (each has its own waits), tails
of one key to a whole tile, groups alone, in second place and far apart, against float64; and the rule of its items."""
import math

import pytest
import torch

from jax_vllm_amd.parts.attention_backend import halves_items

from .test_kernels_gpu import K, _mfma_inputs, _mfma_reference, _prefill_work


def test_the_rule():
    assert halves_items(16, 8, 64, 0, False, 8, 256) == (True, 1)              # few, short
    assert halves_items(350, 175, 256, -256, False, 8, 256) == (True, 1)       # blocks
    assert halves_items(350, 175, 256, 256, False, 8, 256) == (False, 2)       # a sliding window
    assert halves_items(128, 64, 1000, 0, False, 8, 256) == (False, 1)
    assert halves_items(129, 65, 1000, 1024, False, 8, 256) == (False, 2)
    assert halves_items(8, 4, 2048, 0, False, 8, 256) == (False, 2)            # far walks


def test_short_walks_beside_a_round_of_blocks():
    for window in (0, 64, 1024, -64):                                       # groups that are one round: their start alone counts
        assert halves_items(320, 160, 256, window, False, 8, 256) == (True, 1)
    assert halves_items(321, 161, 256, 1024, False, 8, 256) == (False, 2)
    assert halves_items(480, 480, 40, 256, False, 8, 256) == (True, 1)         # requests of one group have no pairs
    assert halves_items(480, 360, 128, 256, False, 8, 256) == (False, 2) and halves_items(480, 361, 128, 256, False, 8, 256) == (True, 1)
    assert halves_items(512, 256, 40, 1024, False, 8, 256) == (False, 2) and halves_items(514, 257, 40, 1024, False, 8, 256) == (True, 1)      # more than a round
    assert halves_items(514, 257, 65, 1024, False, 8, 256) == (False, 2)
    assert [halves_items(512, 256, keys, 1024, False, 4, 256)[0] for keys in (64, 65, 192, 193)] == [True, True, True, False]      # four kv heads
    assert halves_items(80, 40, 257, 0, False, 8, 256) == (False, 1) and halves_items(80, 40, 257, 0, True, 8, 256) == (True, 1)      # a cap
    assert halves_items(300, 150, 400, 0, False, 8, 256) == (True, 1) and halves_items(300, 150, 401, 0, True, 8, 256) == (False, 2)
    assert halves_items(330, 165, 300, 0, True, 8, 256) == (False, 2) and halves_items(330, 165, 300, 0, False, 8, 304) == (True, 1)


def test_a_plan_counts_its_items(monkeypatch):
    """Groups and pairs request by request: 30 prompts of 40 tokens with a q head a kv head have no pair, 16 rows a wave take them."""
    from types import SimpleNamespace

    from jax_vllm_amd.ops import kernels
    from jax_vllm_amd.parts import attention_backend

    monkeypatch.setattr(kernels, "compute_units", lambda device: 256)
    monkeypatch.setattr(attention_backend, "upload_i32", lambda values, device: torch.tensor(values, dtype=torch.int32))
    asked, rule = [], halves_items
    monkeypatch.setattr(attention_backend, "halves_items", lambda *a: asked.append(a) or rule(*a))

    def plan(lens, nq, nkv, **kw):
        ctx = SimpleNamespace(q_lens_host=lens, context_lens_host=[0] * len(lens), page_size=16, block_tables=[torch.zeros(len(lens), 64)])
        return attention_backend.plan_mfma(ctx, nq, nkv, 256, kw.pop("window", 0), "cpu", **kw)

    assert plan([40] * 30, 16, 16, window=1024).one_group and asked[-1] == (480, 480, 40, 1024, False, 16, 256)
    plan([1, 129, 1, 300], 16, 8, capped=True)
    assert asked[-1] == (15 * 8, 8 * 8, 300, 0, True, 8, 256)      # single tokens are no prompt's


@pytest.mark.gpu
@pytest.mark.parametrize("plan", ["single", "second", "neighbours", "far"])
@pytest.mark.parametrize("nq,nkv,reqs,window", [
    (2, 1, [(0, 2), (0, 33), (61, 3), (62, 3), (63, 2)], None),                    # one tile, and one key of a second
    (4, 1, [(126, 2), (127, 2), (190, 3), (255, 40)], None),                       # two, three, four and more
    (16, 1, [(0, 100), (500, 12)], 64),                                            # walks that begin inside a page
    (3, 3, [(40, 300)], 30),                                                       # far groups leave a gap
    (12, 2, [(0, 64), (9, 2), (1017, 30)], 1024),
], ids=str)
def test_walks(nq, nkv, reqs, window, plan):
    d, scale = 256, 1.0 / math.sqrt(256)
    qs, ks, vs, dev = _mfma_inputs(nq, nkv, d, 16, reqs)
    work, n_work = _prefill_work(reqs, nq // nkv, d, window, plan)
    ref = _mfma_reference(qs, ks, vs, reqs, scale, window, nq, d)
    top = max(float(v.abs().max()) for v in vs)
    first = None
    for _ in range(3):
        out = torch.full((dev["n"], nq * d), float("nan"), dtype=torch.bfloat16).cuda()
        K().attn_prefill_mfma(out, dev["q"], dev["stride"], dev["k_pages"], dev["v_pages"], dev["tables"], dev["cu"], dev["ctx"],
                              work, n_work, nq, nkv, d, scale, window or 0)
        # probabilities and results are rounded to 8 bits of fraction: 2^-9 of a weighted sum of values each, at most
        err = float((out.double().cpu() - ref).abs().max())
        assert err <= 2 * 2.0 ** -9 * top + 1e-3, err
        first = out if first is None else first
        assert torch.equal(out, first)
