"""Prefill attention at head size 256 and pages of 16, two waves to 32 rows: walks of one tile to several (each has its own waits), tails
of one key to a whole tile, groups alone, in second place and far apart, against float64; and the rule of its items."""
import math

import pytest
import torch

from jax_vllm_amd.parts.attention_backend import halves_items

from .test_kernels_gpu import K, _mfma_inputs, _mfma_reference, _prefill_work


def test_the_rule():
    assert halves_items(True, 16, 64, 0, 256) == (True, 1)              # few, short
    assert halves_items(True, 350, 256, -256, 256) == (True, 1)         # blocks
    assert halves_items(True, 350, 256, 256, 256) == (False, 2)         # a sliding window
    assert halves_items(True, 128, 1000, 0, 256) == (False, 1)
    assert halves_items(False, 129, 1000, 1024, 256) == (False, 2)
    assert halves_items(False, 8, 2048, 0, 256) == (False, 2)           # far walks


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
