"""Chooses and plans the attention kernels of one step.

bfloat16 with a head size and page size the matrix-core kernels are built for: requests with
one token in the step go to the decode kernel (keys shared out to several blocks when few
requests would leave the chip idle), all others to the prefill kernel in groups of 64 (query,
head-in-group) rows; a work item names two groups of one request, heaviest items first: two
neighbours where the kernel gives each group waves of its own (they see the same keys), else,
while all blocks are on the chip at once, a group that sees many keys with one that sees few, so
that all blocks carry the same load.  float32 with a head size and page size the 32-bit
matrix-core kernel is built for runs that one, in work items of 16 rows.  Everything else
(other head sizes and page sizes) runs the generic float-math kernel.  The plan depends on the
step's lengths, the heads-per-group ratio and which keys the layer's queries see, so it is built
once per step and shared by all layers alike.
"""
from __future__ import annotations

from dataclasses import dataclass
from typing import Optional

import numpy as np
import torch

from ..ops import kernels as K

TARGET_BLOCKS = 256          # blocks of the decode kernel that fill the chip: one per compute unit (measured: 8 requests of
                             # 1,060 keys over 8 kv heads take 13.7 us with 4 splits, 15.5 with 8)
DECODE_TILE = K.ATTN_DECODE_TILE_KEYS      # keys of a tile of the decode kernel; a block has 4 waves with a tile each
RESIDENT_BLOCKS = 2          # blocks of the prefill kernel that a compute unit holds at once


def upload_i32(values, device) -> torch.Tensor:
    """int32 on the device from host integers, through pinned memory."""
    staged = torch.empty(len(values), dtype=torch.int32, pin_memory=True)
    staged.numpy()[:] = values
    return staged.to(device, non_blocking=True)


@dataclass
class MfmaPlan:
    prefill_work: Optional[torch.Tensor]   # int32 [n, 3]
    n_prefill: int
    decode_work: Optional[torch.Tensor]    # int32 [n]; None when the step holds decoded tokens only
    n_decode: int
    num_splits: int
    scratch: Optional[torch.Tensor]
    one_group: bool = False                # prefill items of one group, 16 rows a wave, where the kernel has both forms


def keys_seen(kv_len: int, window: int, keep: int = 0) -> int:
    """The most keys a query sees that has ``kv_len`` keys up to itself (``K.key_window``'s number, and the first keys
    that are kept whatever the window)."""
    return min(kv_len, abs(window) + keep) if window else kv_len


def decode_splits(n_decode: int, blocks_per_request: int, max_kv_len: int) -> int:
    """Blocks that share out a request's keys: as many as give no unit a second block (one more costs a further merge and leaves
    units with twice the load of others: 12 requests of 500 to 1,500 keys over 8 kv heads 18.9 us with 2, 22.2 with 3; 24 of 450 to 1,350
    24.7 with 1, 29.6 with 2; 9 of 500 to 1,500 15.4 with 3, 19.3 with 4).  So also at long contexts, where a merge weighs little (8 kv
    heads, even keys, 1 / 2 splits: 17 requests of 256 keys 10.0 / 14.2, 2,600 40.8 / 50.5, 7,800 111 / 131; 20 of 3,850 61.0 / 71.4; 24 68.0 / 76.0;
    28 78.6 / 81.4; 31 86.8 / 88.8; spread over half to one and a half of that the same but for less).  Open: 3 splits at 17 to 20
    requests of 1,600 spread keys or more (17 of 3,850 60.9, with one 68.3)."""
    base = max(1, n_decode * blocks_per_request)
    tiles = -(-max_kv_len // DECODE_TILE)
    splits = min(max(1, TARGET_BLOCKS // base), splits_by_length(tiles))
    # two blocks spare less than the merge costs while few waves have a third tile (8 kv heads, one request of 300 keys 9.8 alone, 11.3 by
    # two, 9.3 by eight; 16 requests 11.5, 13.4; 16 of 1,100 26.7, 23.8)
    return 1 if splits == 2 and tiles < 24 else splits


def splits_by_length(tiles: int) -> int:
    """How many blocks a request's tiles of keys are worth.  One unit brings in about 48 GB/s whatever a block's waves ask for (1.35 us
    for a tile a wave), so tiles are shared out thinly; the merge takes partial results in batches of 8.  Head size 128, one request
    over 8 kv heads, microseconds with its merge: 150 keys 8.4 by one block, 8.9 by four; 300 keys 9.8 by one, 9.25 by eight; 520 keys
    12.1, by four 10.2, by eight 9.3; 1,024 keys 15.2, 10.2 by eight, 10.7 by sixteen; 2,500 keys 13.7 by eight, 12.2 by sixteen, 12.9 by nineteen;
    7,900 keys 17.3 by sixteen, 16.6 by 24, 17.2 by 32; one over 4 kv heads 15.0 by 32, 17.7 by 61.
    A recorded step is planned for the most keys its block tables hold, a power of two of pages: the plan of 256 keys serves 129 on, that of 2,048 keys
    1,025 on.  What that costs there, attention and output product (2,048 rows), 8 kv heads of 4 q heads: 130 to 250 keys by eight or one block, one request
    14.1 to 15.0 and 13.9 to 14.3, two 14.8 to 15.7 and 14.2 to 14.4, four 15.2 to 16.1 and 14.5 to 14.7; 1,030 to 2,000 keys by sixteen or eight
    15.4 to 16.2 and 15.4 to 16.2, two requests 15.7 to 16.5 and 16.0 to 16.9."""
    return 1 if tiles < 8 else 8 if tiles <= 48 else max(16, tiles // 8)


KEY_TILE = 64                # keys of one tile of the prefill kernel


def prefill_work_items(q_lens, context_lens, g: int, window: int, group_rows: int, groups_per_item: int,
                       balance: bool = True, keep: int = 0):
    """Work items (request, first row of group 0, first row of group 1 or -1) of the prefill kernel
    for the requests with more than one token, heaviest first.  Rows are (query, head-in-group)
    pairs.  ``window``: see ``K.key_window``; ``keep``: first keys every query sees besides.  With ``balance`` and no window the i-th lightest group of a request is paired with its
    i-th heaviest: every pair then walks about the same number of (row tile, key tile) products,
    which matters when the items are so few that the heaviest one decides the time.  Otherwise
    neighbours are paired: they share nearly all their keys, so every fragment read feeds both."""
    items = []
    for r, (ql, cl) in enumerate(zip(q_lens, context_lens)):
        if ql <= 1:
            continue
        groups = []
        if ql * g > 16 * group_rows:       # all groups at once: 512 of them 90 us instead of 350, a few are quicker one by one
            m0 = np.arange(0, ql * g, group_rows)
            end, first = cl + (np.minimum(ql * g, m0 + group_rows) - 1) // g + 1, cl + m0 // g
            begin = np.maximum(0, first - window + 1) if window > 0 else first - first % -window if window else 0 * first
            tiles = -(-end // KEY_TILE) - begin // KEY_TILE + np.minimum(begin // KEY_TILE, -(-keep // KEY_TILE))
            groups = list(zip(tiles.tolist(), m0.tolist()))
        for m0 in range(0, ql * g if not groups else 0, group_rows):
            last_row = min(ql * g, m0 + group_rows) - 1
            end = cl + last_row // g + 1
            first = cl + m0 // g
            begin = max(0, first - window + 1) if window > 0 else first - first % -window if window else 0
            groups.append((-(-end // KEY_TILE) - begin // KEY_TILE + min(begin // KEY_TILE, -(-keep // KEY_TILE)), m0))
        if groups_per_item < 2:
            items.extend((t, r, m0, -1) for t, m0 in groups)
        elif window or not balance:
            for i in range(0, len(groups) - 1, 2):
                items.append((groups[i][0] + groups[i + 1][0], r, groups[i][1], groups[i + 1][1]))
            if len(groups) % 2:
                items.append((groups[-1][0], r, groups[-1][1], -1))
        else:
            lo, hi = 0, len(groups) - 1          # groups are in ascending order of keys seen
            while lo < hi:
                items.append((groups[lo][0] + groups[hi][0], r, groups[hi][1], groups[lo][1]))
                lo, hi = lo + 1, hi - 1
            if lo == hi:
                items.append((groups[lo][0], r, groups[lo][1], -1))
    items.sort(key=lambda w: -w[0])
    return [(r, a, b) for _, r, a, b in items]


def pair_up_resident_items(items: list, first_round: int) -> list:
    """For a launch whose blocks are all on the chip at once, two to a compute unit: the ``first_round`` heaviest
    items (the blocks that get a unit to themselves at first) stay in descending order and the others follow in
    ASCENDING order.  The hardware hands out blocks in the order of their numbers and comes back to the first unit
    after one round, so the unit with the heaviest item gets the lightest one beside it (2,048 tokens, 32 q heads
    over 8 kv heads of 128: 53.9 against 58.3 us; with more items than fit at once, heaviest first stays the
    rule: 94.8 against 103.3 us at 3,072)."""
    return items[:first_round] + items[first_round:][::-1]


def prefill_item_shape(rows: int, nkv: int, group_rows: int, kernel_groups: int, compute_units: int,
                       waves_split: bool = False):
    """(groups per work item, whether light groups are paired with heavy ones) for a step with
    ``rows`` (query, head-in-group) rows per kv head in its prompt portions.  A kernel whose groups
    have waves of their own (``waves_split``) always gets neighbouring pairs: half of a block's waves
    would idle through the keys that only one group sees (2,048 tokens, 32 q heads over 8 kv heads
    of 128: 64 against 78 us; one group per item: 88).  For the other kernel, measured on the same
    heads: while items of two groups would not even give every compute unit a block,
    items of one group do better although every block then loads its keys for half the rows
    (512 tokens after 3,000: 111 against 135 us; after 16,000: 507 against 622); balancing wins
    while all blocks are on the chip at once, two per compute unit (2,048 tokens, 512 blocks: 88
    against 98 us); one more block and the equal loads need a whole further round, so neighbours
    that share their keys, heaviest first, win from there (2,304 tokens, 576 blocks: 111 against
    137 us; 8,192: 887 against 1,036)."""
    if waves_split:
        return kernel_groups, False
    blocks = -(-rows // (group_rows * kernel_groups)) * nkv
    if kernel_groups > 1 and blocks <= compute_units:
        return 1, True
    return kernel_groups, blocks <= RESIDENT_BLOCKS * compute_units


def few_rows_of_256(rows: int, group_rows: int, compute_units: int) -> bool:
    """Whether a step's prompt portions at head size 256 and pages of other than 16 keys take items of one group (16 rows a wave) instead of two (32): while those
    give no more than a quarter of the compute units a second block, whatever the keys, for the larger form has no work of its own to overlap there.  Microseconds, two groups /
    one: 512 tokens after 4,000, 16 heads over one, with pages of 32 203 / 192, of 24 259 / 209; 2,048 over 8 kv heads with pages of 32 98 / 93.  (Pages of 16:
    ``halves_items``.)"""
    return 4 * -(-rows // group_rows) <= 5 * compute_units


SHORT_WALK = 400             # keys up to which the halves kernel's start weighs as much as its tiles


def halves_items(groups: int, pairs: int, keys: int, window: int, capped: bool, kv_heads: int, compute_units: int):
    """(Whether 16 rows a wave take them, groups per item) at head size 256 and pages of 16 keys, where two waves share 32 rows of the
    other form.  ``groups``, ``pairs``: items of one group and of two (neighbours of one request) that the prompts have over all kv heads; ``keys``: the most that a
    query sees; ``capped``: scores go through a cap, which is paid once more for every wave that starts.

    Walks of more than 400 keys: the halves, by pairs once groups alone give half of the compute units a block or the walk is far (no slower then, and half
    the reads).  Shorter ones: the 16 rows a wave, whose start is short, while the groups are a round of blocks (a quarter of the units a second one), but items of one
    group where 257 keys and more are scored without a cap and no unit has two; beyond a round the pairs, if the prompts have them (a request of one group has
    none), where a sliding window or 257 keys bound the walk, and up to 64 keys, a tile, only if they are one round.  Four kv heads, two dies to a head: not up to 192
    keys, where the halves take some 14 us more than with other counts (8 heads over 4, whatever the strides and the order of pages; why is not known).  Microseconds, 16 rows a wave /
    items of one group / of two: 16 heads over one, 64 tokens 10.1 / 10.7 / 13.9, 300 20.6 / 20.1 / 22.0, with a cap 22.3 / 22.8 / 24.7, 512 28.6 / 26.3 / 27.3, 1,000 50.5 /
    45.4 / 43.4, with a window of 100 16.6 / - / 20.1, 2,048 with a window of 1,024 104 / 91 / 51, of 256 44 / 43 / 27, of 128 33 / 33 / 23; 512 after
    4,000 193 / 154 / 155; 30 prompts of 40 tokens, 8 heads over one 10.5 / 11.9 / 15.4, 16 over 8 18.3 / 20.6 / 14.2, 60 of them, 16 over one 29.5 / 33.5 / 31.7; 4,096
    tokens of 8 heads over 4 with a window of 128 33.8 / 34.0 / 38.6, of 32 25.2 / 43.5 / 38.2, of 256 44 / 45 / 41, 2,048 of 16 over 8 with 128 33.1 / 33.3 / 25.4.  Of 2,300
    steps that the 16 rows a wave took before (16 head layouts, 27 sets of prompts, windows of 32 to 1,024, blocks, with and without a cap) none takes more than 1.02 of their time."""
    if keys > SHORT_WALK:
        return False, 2 if 2 * groups > compute_units or keys >= 2048 else 1
    if 4 * groups <= 5 * compute_units:
        return keys <= 256 or capped or groups > compute_units, 1
    if (keys <= 256 and window <= 0) or 4 * pairs > 3 * groups:
        return True, 1
    if keys <= KEY_TILE and pairs > compute_units or keys <= 3 * KEY_TILE and kv_heads == 4:
        return True, 1
    return False, 2


def plan_mfma(ctx, nq: int, nkv: int, head_dim: int, window: int, device, keep: int = 0, capped: bool = False) -> MfmaPlan:
    g = nq // nkv
    group_rows, kernel_groups = K.attn_prefill_geometry(head_dim)
    rows = sum(ql * g for ql in ctx.q_lens_host if ql > 1)
    groups_per_item, balance = prefill_item_shape(rows, nkv, group_rows, kernel_groups, K.compute_units(device),
                                                  K.attn_prefill_waves_split(head_dim))
    cus = K.compute_units(device)
    one_group = False
    if head_dim == 256:
        if ctx.page_size == 16:
            keys = max([keys_seen(cl + ql, window, keep) for ql, cl in zip(ctx.q_lens_host, ctx.context_lens_host) if ql > 1], default=0)
            groups = [-(-ql * g // group_rows) for ql in ctx.q_lens_host if ql > 1]
            pairs = sum((n + 1) // 2 for n in groups) * nkv
            one_group, groups_per_item, balance = *halves_items(sum(groups) * nkv, pairs, keys, window, capped, nkv, cus), False
        elif few_rows_of_256(rows * nkv, group_rows, cus):
            one_group, groups_per_item, balance = True, 1, False
    prefill = prefill_work_items(ctx.q_lens_host, ctx.context_lens_host, g, window, group_rows, groups_per_item,
                                 balance=balance, keep=keep)
    # head size 256: items of two groups have a unit each, and items of one group were not helped (168 steps of 257 to 512 items, all
    # page sizes: 0.97 to 1.24 of the time, 1.04 on average)
    if cus < len(prefill) * nkv <= RESIDENT_BLOCKS * cus and head_dim != 256:
        prefill = pair_up_resident_items(prefill, cus // nkv)
    decode = [r for r, ql in enumerate(ctx.q_lens_host) if ql == 1]
    max_kv_decode = max([ctx.context_lens_host[r] + 1 for r in decode], default=1)
    splits = decode_splits(len(decode), nkv * (-(-g // 16)), keys_seen(max_kv_decode, window, keep)) if decode else 1
    if decode:      # a very wide block table is taken split by split
        widest = max(t.shape[1] for t in ctx.block_tables)
        splits = max(splits, K.attn_decode_min_splits(widest, ctx.page_size, keep))
    decode_only = len(decode) == len(ctx.q_lens_host)       # requests 0, 1, ...: the kernel needs no list
    flat = [x for item in prefill for x in item] + ([] if decode_only else decode)
    dev = upload_i32(flat, device) if flat else None
    n_pre = len(prefill)
    scratch = None
    if decode and splits > 1:
        scratch = torch.empty(K.attn_decode_scratch_floats(len(decode), nq, splits, head_dim),
                              dtype=torch.float32, device=device)
    return MfmaPlan(dev[: 3 * n_pre] if n_pre else None, n_pre,
                    dev[3 * n_pre:] if decode and not decode_only else None, len(decode), splits, scratch, one_group)


@dataclass
class F32Plan:
    work: torch.Tensor               # int32 [n, 2]
    n_work: int
    splits: int
    parts: Optional[torch.Tensor]


def f32_work_items(q_lens, context_lens, g: int, rows: int):
    """Work items (request, first row) of the 32-bit kernel, those that see the most keys first."""
    items = [(-(cl + -(-min(ql * g, m0 + rows) // g)), r, m0)
             for r, (ql, cl) in enumerate(zip(q_lens, context_lens)) for m0 in range(0, ql * g, rows)]
    return [(r, m0) for _, r, m0 in sorted(items)]


def f32_ranges(kv_len: int, window: int, keep: int, rows: int, range_keys: int) -> int:
    """The most ranges of keys that a work item of the 32-bit kernel touches: its ``rows`` rows are queries next to one another,
    the last at ``kv_len`` - 1 at most.  (An interval of n keys touches up to (n + size - 2) / size + 1 ranges.)"""
    whole = -(-kv_len // range_keys)
    if not window:
        return whole
    return min(whole, -(-keep // range_keys) + (abs(window) + rows - 1 + range_keys - 2) // range_keys + 1)


def plan_f32(ctx, nq: int, nkv: int, head_dim: int, window: int, device, keep: int) -> F32Plan:
    rows = K.attn_f32_rows()
    items = f32_work_items(ctx.q_lens_host, ctx.context_lens_host, nq // nkv, rows)
    most = max(c + q for c, q in zip(ctx.context_lens_host, ctx.q_lens_host))
    size = K.attn_f32_range_keys()
    # keys that fit a range: nothing to share out, though they may touch two
    ranges = f32_ranges(most, window, keep, rows, size) if keys_seen(most, window, keep) > size else 1
    splits = K.attn_f32_splits(len(items), nkv, ranges, device)
    parts = None
    if splits > 1:
        parts = torch.empty(K.attn_f32_part_floats(len(items), nkv, ranges, head_dim), dtype=torch.float32, device=device)
    return F32Plan(upload_i32([x for item in items for x in item], device), len(items), splits, parts)


def token_possible(att, ctx, mem, interleaved: bool, rotary_dim: int) -> bool:
    """Whether a step of single tokens goes from the q/k/v product to its attention in one launch (``run_token``)."""
    return (ctx.decode_only and mem.writes and not getattr(att, "softcap", None) and not getattr(att, "keep_first", 0)
            and K.attn_decode_token_possible(att.dtype, att.d, ctx.page_size, interleaved, rotary_dim, att.rotation is not None))


TOKEN_GROUP = 6              # q heads of a kv head that a block prepares with its new key and value in one round of loads (4 waves, 2 heads each)
TOKEN_BLOCKS = 2048          # (request, kv head) pairs from which on a block's start has to be short beside its keys


def token_pays(att, ctx) -> bool:
    """Whether that launch had better stand for the two it replaces, which prepare a head once and not in every block that reads it.  Up to 6 q heads of a kv
    head: two launches' time over one's, 396 steps of 1 to 256 requests of 30 to 3,000 keys, 1 to 32 kv heads, 0.99 to 1.24, 1.09 on average.  More heads a
    group come in further rounds of loads (8: 0.92 to 1.16, from 64 requests on 0.94 and more; 16: 0.75 to 1.35, 0.95 on average), and 2,048 pairs or more of
    a request and a kv head with few keys queue up behind that start (256 requests over 8 kv heads 30 keys 0.88, 200 keys 0.98, 400 1.02; 128 over 32 0.89 to 0.99)."""
    return att.nq // att.nkv <= TOKEN_GROUP and (
        ctx.num_tokens * att.nkv < TOKEN_BLOCKS or keys_seen(ctx.max_kv_len, K.key_window(att.window, att.chunk)) >= 1024)


def _mfma_plan(att, ctx, window: int, keep: int, device) -> MfmaPlan:
    capped = att.d == 256 and bool(getattr(att, "softcap", None))      # (nothing else of a plan depends on a cap)
    key = ("mfma_attention_plan", att.nq, att.nkv, att.d, window, keep, capped)
    plan = ctx.plans.get(key)
    if plan is None:
        plan = ctx.plans[key] = plan_mfma(ctx, att.nq, att.nkv, att.d, window, device, keep, capped)
    return plan


def _decode_work(ctx, plan, att, window: int):
    """The order of a step's decoding requests: the plan's list, or by their lengths where a step of single tokens gives units blocks of more than
    one request and 512 keys or more (shorter ones differ by less than the look-up takes)."""
    heads = att.nkv * (-(-(att.nq // att.nkv) // 16))
    at_once = TARGET_BLOCKS // heads
    if (not ctx.decode_only or plan.num_splits > 1 or not 0 < at_once < plan.n_decode <= K.DECODE_ORDER_MAX
            or keys_seen(ctx.max_kv_len, window) < 512):
        return plan.decode_work
    key = ("decode_order", at_once, window)      # a result of the device: made anew in every step, also a replayed one
    if key not in ctx.extras:
        ctx.extras[key] = K.decode_order(ctx.context_lens, at_once, window)
    return ctx.extras[key]


def run_token(att, qkv, cos_sin, rotary_dim: int, ctx, mem, whole: bool = False):
    """Head norms, rotation, page writes and attention of a step of single tokens; ``qkv``: the q/k/v product or its parts.  Returns the
    heads [tokens, nq * D], or ``K.SplitHeads`` where the output product merges them (``whole``: never)."""
    window = K.key_window(att.window, att.chunk)
    n, device = ctx.num_tokens, att.w_o.device
    plan = _mfma_plan(att, ctx, window, 0, device)
    merge = whole or plan.num_splits == 1 or not K.split_heads_pay(n, att.w_o, plan.num_splits)
    out = torch.empty((n, att.nq * att.d), dtype=att.dtype, device=device) if merge else None
    K.attn_decode_token(out, qkv, ctx.slot_mappings[mem.group], att.q_norm, att.k_norm, att.qk_norm_eps or 0.0, cos_sin, rotary_dim,
                        mem.pages["k"], mem.pages["v"], ctx.block_tables[mem.group], ctx.context_lens, att.nq, att.nkv, att.d,
                        att.scale, window, plan.num_splits, plan.scratch, sinks=att.sinks, merge=merge, work=_decode_work(ctx, plan, att, window))
    return out if merge else K.SplitHeads(plan.scratch, n, plan.num_splits, att.nq, att.d, att.sinks)


def run(att, out, qkv, ctx, mem, terms: "bool | None" = None):
    """Attention of the step's tokens into ``out``; returns it, or ``K.TermRows`` where ``terms`` (``K.f32_terms_layout`` of the product that reads it)
    asks for them and one block makes a row."""
    # q heads of a row sit at the front of the fused q/k/v projection, unless the mixer says where else
    q_row_stride = getattr(att, "q_row_stride", None) or (att.nq + 2 * att.nkv) * att.d
    window = K.key_window(att.window, getattr(att, "chunk", None))
    sinks = getattr(att, "sinks", None)      # float [nq] or None: one more term exp(sink) in every softmax denominator
    cap = getattr(att, "softcap", None) or 0.0                       # scores under a soft cap
    keep = (getattr(att, "keep_first", 0) or 0) if window else 0     # first keys seen whatever the window
    if K.attn_f32_possible(qkv.dtype, att.d, ctx.page_size):
        key = ("attn_f32_plan", att.nq, att.nkv, att.d, window, keep)
        plan = ctx.plans.get(key)
        if plan is None:
            plan = ctx.plans[key] = plan_f32(ctx, att.nq, att.nkv, att.d, window, qkv.device, keep)
        left = K.f32_terms(out.shape[0], out.shape[1], terms, out.device) if terms is not None and plan.splits == 1 else None
        K.attn_f32(out, qkv, q_row_stride, mem.pages["k"], mem.pages["v"], ctx.block_tables[mem.group], ctx.cu_seqlens,
                   ctx.context_lens, plan.work, plan.n_work, att.nq, att.nkv, att.d, att.scale, window, plan.splits,
                   plan.parts, sinks=sinks, cap=cap, keep=keep, terms=None if left is None else (left, terms))
        return out if left is None else K.TermRows(out, left, terms)
    if not K.mfma_attention_supported(qkv.dtype, att.d, ctx.page_size):
        K.paged_attention_generic(
            out, qkv, q_row_stride, mem.pages["k"], mem.pages["v"], ctx.block_tables[mem.group], ctx.token_req,
            ctx.positions, att.nq, att.nkv, att.d, att.scale, window, sinks=sinks, cap=cap, keep=keep,
        )
        return out
    plan = _mfma_plan(att, ctx, window, keep, qkv.device)
    tables = ctx.block_tables[mem.group]
    if (plan.n_prefill and plan.n_decode and not cap and not keep and not plan.one_group
            and K.attn_mixed_possible(att.d, ctx.page_size, tables.shape[1], att.nq, att.nkv)):
        K.attn_mixed(out, qkv, q_row_stride, mem.pages["k"], mem.pages["v"], tables, ctx.cu_seqlens, ctx.context_lens, plan.prefill_work,
                     plan.n_prefill, _decode_work(ctx, plan, att, window), plan.n_decode, att.nq, att.nkv, att.d, att.scale, window,
                     plan.num_splits, plan.scratch, sinks=sinks)
        return out
    if plan.n_prefill:
        K.attn_prefill_mfma(out, qkv, q_row_stride, mem.pages["k"], mem.pages["v"], tables, ctx.cu_seqlens,
                            ctx.context_lens, plan.prefill_work, plan.n_prefill, att.nq, att.nkv, att.d, att.scale,
                            window, sinks=sinks, cap=cap, keep=keep, one_group=plan.one_group)
    if plan.n_decode:
        K.attn_decode_mfma(out, qkv, q_row_stride, mem.pages["k"], mem.pages["v"], tables, ctx.cu_seqlens,
                           ctx.context_lens, _decode_work(ctx, plan, att, window), plan.n_decode, att.nq, att.nkv, att.d, att.scale,
                           window, plan.num_splits, plan.scratch, sinks=sinks, cap=cap, keep=keep)
    return out
