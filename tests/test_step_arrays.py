"""What the host makes at once for a step (its arrays, its prompts' work list, its token checks) against the
same made token by token and group by group."""
import numpy as np
import pytest
import torch

from jax_vllm_amd.cache import CacheManager
from jax_vllm_amd.engine.core import EngineCore
from jax_vllm_amd.engine.entries import StepEntry
from jax_vllm_amd.parts.attention_backend import KEY_TILE, prefill_work_items

PAGE = 16


def _core(groups, vocab=1000):
    core = object.__new__(EngineCore)
    core.vocab_size, core.page_size, core.device, core.group_keys = vocab, PAGE, torch.device("cpu"), groups
    core.cache = CacheManager(groups, PAGE, 64, 8)
    return core


def _entries(core, contexts, portions, rng):
    entries = []
    for i, (context, ql) in enumerate(zip(contexts, portions)):
        rid = f"r{i}"
        core.cache.start(rid)
        for n in [8] * (context // 8) + [context % 8]:       # pages outside a window leave the table on the way
            if n:
                core.cache.reserve(rid, n)
                core.cache.commit(rid, rng.integers(0, 1000, n).tolist())
        core.cache.reserve(rid, ql)
        entries.append(StepEntry(rid, rng.integers(0, 1000, ql).tolist(), [0, ql - 1] if i % 2 else [ql - 1]))
    return entries


@pytest.mark.parametrize("groups", [[("full",)], [("full",), ("window", 20)], [("window", 20), ("chunk", 24)]])
@pytest.mark.parametrize("contexts,portions", [([0], [1]), ([0], [2]), ([37, 0, 16, 5], [1, 33, 16, 3]), ([100, 15, 0], [1, 1, 1])])
def test_arrays_of_a_step_equal_those_made_token_by_token(groups, contexts, portions, monkeypatch):
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, pin_memory=False, **k: empty(*a, **k))       # no device here to pin for
    core = _core(groups)
    entries = _entries(core, contexts, portions, np.random.default_rng(7))
    tokens, ctx, rows = core._build(entries, core._checked_tokens(entries))

    want = {name: [] for name in ("tok", "prev", "pos", "req", "rows")}
    slots, cu = [[] for _ in groups], [0]
    for i, e in enumerate(entries):
        n, before = len(e.tokens), core.cache.context_len(e.request_id)
        want["rows"] += [cu[-1] + w for w in e.want]
        want["tok"] += e.tokens
        want["prev"] += [core.cache.last_token(e.request_id)] + e.tokens[:-1]
        want["pos"] += range(before, before + n)
        want["req"] += [i] * n
        cu.append(cu[-1] + n)
        for g in range(len(groups)):
            slots[g] += core.cache.slot_mapping(e.request_id, g, n)
    got = {"tok": tokens, "prev": ctx.prev_tokens, "pos": ctx.positions, "req": ctx.token_req, "rows": rows}
    assert {k: v.tolist() for k, v in got.items()} == want
    assert ctx.cu_seqlens.tolist() == cu and ctx.context_lens.tolist() == contexts
    assert ctx.slot_ids.tolist() == [core.cache.slot(e.request_id) for e in entries]
    assert [m.tolist() for m in ctx.slot_mappings] == slots
    for g, table in enumerate(ctx.block_tables):
        for row, e in zip(table.tolist(), entries):
            pages = core.cache.block_table(e.request_id, g)
            assert row == pages + [0] * (table.shape[1] - len(pages))


def test_a_token_without_a_page_is_named(monkeypatch):
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, pin_memory=False, **k: empty(*a, **k))
    core = _core([("full",)])
    entries = _entries(core, [20, 3], [4, 20], np.random.default_rng(7))
    core.cache.block_table("r1", 0)[1] = 0
    with pytest.raises(RuntimeError, match="'r1': position 16 has no page"):
        core._build(entries, core._checked_tokens(entries))


def test_tokens_of_every_integer_form_are_taken():
    core = _core([("full",)])
    forms = [[1, 2, 3], (1, 2, 3), np.array([1, 2, 3]), np.array([1, 2, 3], dtype=np.uint8), np.array([1, 2, 3], dtype=np.uint64),
             torch.tensor([1, 2, 3]), [np.int32(1), 2, torch.tensor(3)], [1.0, 2.0, 3.0], [True, 2, 3]]
    for form in forms:
        ids = core._checked_tokens([StepEntry("a", form, [2]), StepEntry("b", [0, 999], [])])
        assert ids.dtype.kind in "iu" and ids.tolist() == [1, 2, 3, 0, 999]


@pytest.mark.parametrize("tokens,want,message", [
    ([5, 1000], [], "token id 1000 outside the vocabulary"), ([-1], [], "token id -1 outside"),
    ([2 ** 40], [], "outside the vocabulary"), ([2 ** 70], [], "outside the vocabulary"), (np.array([2 ** 63], dtype=np.uint64), [], "outside"),
    ([1, 2], [2], "wanted place 2 outside its 2 tokens"), ([1, 2], [-1], "wanted place -1 outside")])
def test_tokens_and_places_outside_are_named(tokens, want, message):
    core = _core([("full",)])
    with pytest.raises(ValueError, match=f"request 'bad': .*{message}"):
        core._checked_tokens([StepEntry("good", [1, 2, 3], [0, 2]), StepEntry("bad", tokens, want)])


def test_tokens_that_are_no_numbers_are_refused():
    with pytest.raises((TypeError, ValueError)):
        _core([("full",)])._checked_tokens([StepEntry("a", ["x"], [])])
    with pytest.raises(TypeError):
        _core([("full",)])._checked_tokens([StepEntry("a", [None], [])])


@pytest.mark.parametrize("window,keep", [(0, 0), (100, 0), (100, 70), (1, 0), (-96, 0), (-96, 70)])
@pytest.mark.parametrize("per_item", [1, 2])
def test_work_lists_made_at_once_equal_those_made_group_by_group(window, keep, per_item):
    """A request of more than 16 groups has them weighed at once."""
    for g, rows, ql, context in [(4, 64, 257, 0), (1, 64, 1025, 37), (5, 32, 200, 1000), (20, 64, 52, 3), (8, 16, 40, 63)]:
        assert ql * g > 16 * rows
        weights = []
        for m0 in range(0, ql * g, rows):
            last = (min(ql * g, m0 + rows) - 1) // g
            first = context + m0 // g
            begin = max(0, first - window + 1) if window > 0 else first - first % -window if window else 0
            weights.append((-(-(context + last + 1) // KEY_TILE) - begin // KEY_TILE + min(begin // KEY_TILE, -(-keep // KEY_TILE)), m0))
        if per_item == 1:
            pairs = [(t, m0, -1) for t, m0 in weights]
        elif window:
            pairs = [(weights[i][0] + (weights[i + 1][0] if i + 1 < len(weights) else 0), weights[i][1],
                      weights[i + 1][1] if i + 1 < len(weights) else -1) for i in range(0, len(weights), 2)]
        else:
            n = len(weights)
            pairs = [(weights[i][0] + weights[n - 1 - i][0], weights[n - 1 - i][1], weights[i][1]) for i in range(n // 2)]
            pairs += [(weights[n // 2][0], weights[n // 2][1], -1)] if n % 2 else []
        pairs.sort(key=lambda p: -p[0])
        assert prefill_work_items([ql], [context], g, window, rows, per_item, keep=keep) == [(0, a, b) for _, a, b in pairs]
