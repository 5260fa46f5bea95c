"""Head norms, rotation, page writes and attention of a step of single tokens in one launch, against the formulas in float64 and
against the two launches it replaces; and the rule that shares a request's keys out to blocks."""
import math

import pytest
import torch

from jax_vllm_amd.parts.attention_backend import decode_splits

D = 128


def test_decode_splits_by_length():
    assert [decode_splits(1, 8, keys) for keys in (1, 224, 225, 1536, 1537, 4096, 8000)] == [1, 1, 8, 8, 16, 16, 31]
    assert [decode_splits(n, 8, 300) for n in (5, 8, 10, 11, 16)] == [6, 4, 3, 1, 1]       # two blocks only from 24 tiles on
    assert [decode_splits(16, 8, keys) for keys in (736, 737, 5000)] == [1, 2, 2]
    for n in range(1, 300):
        for keys in (1, 31, 200, 1000, 30000):
            assert n * 8 * decode_splits(n, 8, keys) <= max(256, n * 8)


CASES = [
    # nq, nkv, page_size, contexts, window, parts (0: bf16 rows), norm, rotated, splits
    (32, 8, 16, [1023, 0, 31, 500], None, 4, True, True, 1),
    (32, 8, 16, [1023, 0, 31, 500], None, 2, True, True, 8),
    (8, 8, 8, [1, 32, 33, 127, 128], None, 3, True, True, 2),
    (12, 2, 24, [95, 96, 200], None, 1, False, True, 5),
    (32, 2, 16, [64, 700], None, 4, True, True, 3),            # 16 heads a group: more rows than are asked for at once
    (40, 2, 16, [77, 300], None, 2, True, True, 2),            # 20 heads a group: two row tiles a kv head, one writes the key
    (4, 1, 32, [40, 2000], 50, 4, True, False, 4),
    (16, 4, 16, [300, 18], -64, 0, True, True, 1),
    (16, 4, 16, [300, 18, 63], None, 0, False, False, 3),
    (16, 4, 16, [64, 128, 0, 63], -64, 2, True, True, 1),      # the first position of a block of positions: its own key alone, no page is read
    (16, 4, 16, [64, 130, 7], -64, 0, True, True, 3),
    (8, 2, 16, [40, 64, 0, 31], 1, 4, True, True, 1),          # a window of the own key alone
    (8, 2, 16, [40, 64, 33], 1, 0, False, True, 4),
    (4, 1, 8, [32900, 5], None, 2, True, True, 3),             # a table row of more entries than a block keeps: only its own split's are copied
]


@pytest.mark.gpu
@pytest.mark.parametrize("sinks", [False, True])
@pytest.mark.parametrize("case", CASES, ids=[f"h{c[0]}g{c[1]}p{c[2]}w{c[4]}n{c[5]}s{c[8]}" for c in CASES])
def test_token_attention_from_the_product(case, sinks):
    from jax_vllm_amd.ops import kernels as K

    nq, nkv, ps, contexts, window, n_parts, norm, rotated, splits = case
    n, width, bf, eps, scale = len(contexts), (nq + 2 * nkv) * D, torch.bfloat16, 1e-6, 1 / math.sqrt(D)
    g = torch.Generator().manual_seed(nq + sum(contexts))
    src = torch.randn(max(1, n_parts), n, width, generator=g)
    if n_parts == 0:
        src = src.to(bf).float()
    pages = sum(c // ps + 1 for c in contexts) + 1
    kp, vp = (torch.randn(pages, nkv, *shape, generator=g).to(bf) for shape in ((ps, D), (D, ps)))
    kp[0] = vp[0] = 0
    order = (torch.randperm(pages - 1, generator=g) + 1).to(torch.int32)
    tables, slots, at = torch.zeros(n, max(contexts) // ps + 3, dtype=torch.int32), [], 0
    for i, c in enumerate(contexts):
        tables[i, :c // ps + 1] = order[at:at + c // ps + 1]
        at += c // ps + 1
        slots.append(int(tables[i, c // ps]) * ps + c % ps)
        vp[int(tables[i, c // ps]), :, :, c % ps:] = float("nan")          # what the cache holds behind the last key counts for nothing
        kp[int(tables[i, c // ps]), :, c % ps:] = float("nan")
    slots[-1] = -1                                                          # a token that is not stored
    qw, kw = ((1 + 0.1 * torch.randn(D, generator=g)) if norm else None for _ in "qk")
    sink = torch.randn(nq, generator=g) if sinks else None
    pos = torch.tensor(contexts, dtype=torch.int32).cuda()
    table = K.rope_table(pos, (1e6 ** (-torch.arange(0, D, 2).float() / D)).cuda()) if rotated else None
    dev = lambda t: None if t is None else t.cuda()
    kc, vc, tc, sc, qwc, kwc = dev(kp), dev(vp), dev(tables), torch.tensor(slots, dtype=torch.int32).cuda(), dev(qw), dev(kw)
    given = (src if n_parts else src[0].to(bf)).cuda()
    out = torch.full((n, nq * D), float("nan"), dtype=bf).cuda()
    scratch = torch.full((max(1, K.attn_decode_scratch_floats(n, nq, splits, D)),), float("nan")).cuda()
    K.attn_decode_token(out, given, sc, qwc, kwc, eps, table, D if rotated else 0, kc, vc, tc, pos, nq, nkv, D, scale, window or 0,
                        splits, scratch, sinks=dev(sink))

    # the formulas; heads are bfloat16 once they are prepared (2^-9 of a head's largest element)
    x = src.double().sum(0).view(n, nq + 2 * nkv, D)
    heads = []
    for part, w in ((x[:, :nq], qw), (x[:, nq:nq + nkv], kw)):
        if w is not None:
            part = part * torch.rsqrt((part * part).mean(-1, keepdim=True) + eps) * w.double()
        if rotated:
            cos, sin = table.double().cpu()[:, None].split(D // 2, -1)
            a, b = part.split(D // 2, -1)
            part = torch.cat([a * cos - b * sin, b * cos + a * sin], -1)
        heads.append(part.to(bf).double())
    q, k, v = *heads, x[:, nq + nkv:].to(bf).double()
    want = torch.zeros(n, nq, D, dtype=torch.float64)
    for i, c in enumerate(contexts):
        idx = [(int(tables[i, j // ps]), j % ps) for j in range(c)]
        ks = torch.stack([kp[p, :, s].double() for p, s in idx] + [k[i]])                # [keys, nkv, D]
        vs = torch.stack([vp[p, :, :, s].double() for p, s in idx] + [v[i]])
        first = 0 if not window else max(0, c - window + 1) if window > 0 else c - c % -window
        for h in range(nq):
            s = ks[first:, h // (nq // nkv)] @ q[i, h] * scale
            if sinks:
                s = torch.cat([s, sink[h].double()[None]])
            want[i, h] = torch.softmax(s, 0)[:c + 1 - first] @ vs[first:, h // (nq // nkv)]
    # weights and results are bfloat16: 2^-8 of either, and a unit of 2^-8 where a prepared head rounds the other way
    torch.testing.assert_close(out.double().cpu().view(n, nq, D), want, rtol=2e-2, atol=2e-2)
    got_k, got_v = kc.cpu(), vc.cpu()
    for i, s in enumerate(slots):
        if s >= 0:
            torch.testing.assert_close(got_k[s // ps, :, s % ps].double(), k[i], rtol=2 ** -7, atol=1e-6)
            torch.testing.assert_close(got_v[s // ps, :, :, s % ps].double(), v[i], rtol=2 ** -7, atol=1e-6)
            kp[s // ps, :, s % ps], vp[s // ps, :, :, s % ps] = got_k[s // ps, :, s % ps], got_v[s // ps, :, :, s % ps]
    same = lambda a, b: torch.equal(a.view(torch.int16), b.view(torch.int16))
    assert same(got_k, kp) and same(got_v, vp)                              # nothing else was written

    # the two launches
    k2, v2 = dev(kp), dev(vp)
    qkv = torch.zeros(n, width, dtype=bf).cuda() if n_parts > 1 else src.sum(0).to(bf).cuda()
    K.qk_norm_rope_write(qkv, sc, qwc, kwc, eps, table, D if rotated else 0, False, k2, v2, ps, nq, nkv, D,
                         parts=given if n_parts > 1 else None)
    out2 = torch.empty_like(out)
    K.attn_decode_mfma(out2, qkv, width, k2, v2, tc, torch.arange(n + 1, dtype=torch.int32).cuda(), pos, None, n, nq, nkv, D, scale,
                       window or 0, splits, scratch, sinks=dev(sink))
    torch.testing.assert_close(out[:-1].float(), out2[:-1].float(), rtol=2e-2, atol=2e-2)      # the last token's key is in no page


@pytest.mark.gpu
def test_token_attention_refuses_what_it_does_not_take():
    from jax_vllm_amd.ops import kernels as K

    possible = K.attn_decode_token_possible
    assert possible(torch.bfloat16, 128, 16, False, 128, True) and possible(torch.bfloat16, 128, 16, False, 0, False)
    assert not possible(torch.float32, 128, 16, False, 128, True) and not possible(torch.bfloat16, 64, 16, False, 64, True)
    assert not possible(torch.bfloat16, 128, 16, True, 128, True) and not possible(torch.bfloat16, 128, 16, False, 64, True)
    assert not possible(torch.bfloat16, 128, 4, False, 128, True)
    bf = dict(dtype=torch.bfloat16, device="cuda")
    i32 = lambda *s: torch.zeros(*s, dtype=torch.int32, device="cuda")
    args = lambda rows: (torch.empty(1, 4 * D, **bf), rows, i32(1), None, None, 0.0, None, 0, torch.zeros(2, 1, 16, D, **bf),
                         torch.zeros(2, 1, D, 16, **bf), i32(1, 1), i32(1), 4, 1, D, 1.0)
    with pytest.raises(K.KernelArgumentError, match="parts"):
        K.attn_decode_token(*args(torch.zeros(5, 1, 6 * D, device="cuda")))
    with pytest.raises(K.KernelArgumentError, match="or parts of that"):
        K.attn_decode_token(*args(torch.zeros(1, 5 * D, **bf)))
    with pytest.raises(K.KernelArgumentError, match="scratch"):
        K.attn_decode_token(*args(torch.zeros(1, 6 * D, **bf)), num_splits=2)


@pytest.mark.gpu
def test_unmerged_splits_lie_by_request():
    """The splits' results that a product merges: those of row r belong to request r, so no order of the blocks goes with them."""
    from jax_vllm_amd.ops import kernels as K

    n, nq, nkv, ps, splits = 3, 4, 1, 16, 2
    g = torch.Generator().manual_seed(5)
    qkv = torch.randn(n, (nq + 2 * nkv) * D, generator=g).to(torch.bfloat16).cuda()
    kp, vp = (torch.randn(1 + 4 * n, nkv, *s, generator=g).to(torch.bfloat16).cuda() for s in ((ps, D), (D, ps)))
    tables = (1 + torch.arange(4 * n, dtype=torch.int32)).view(n, 4).cuda()
    pos = torch.tensor([60, 3, 41], dtype=torch.int32).cuda()
    slots = (tables[torch.arange(n), (pos // ps).long()] * ps + pos % ps).to(torch.int32)
    work = torch.tensor([2, 0, 1], dtype=torch.int32).cuda()

    def attend(merge, order):
        scratch = torch.full((K.attn_decode_scratch_floats(n, nq, splits, D),), float("nan")).cuda()
        out = torch.full((n, nq * D), float("nan"), dtype=torch.bfloat16).cuda()
        K.attn_decode_token(out if merge else None, qkv, slots, None, None, 0.0, None, 0, kp, vp, tables, pos, nq, nkv, D, 1.0, 0, splits, scratch,
                            merge=merge, work=order)
        return out, scratch

    out, scratch = attend(True, None)
    assert torch.equal(attend(True, work)[0], out)                 # merged, any order
    kept = attend(False, None)[1]
    acc, ml = kept[:n * nq * splits * D].view(n, nq, splits, D), kept[n * nq * splits * D:].view(n, nq, splits, 2)
    f = torch.exp2(ml[..., 0] - ml[..., 0].amax(-1, keepdim=True))
    merged = (torch.where(f[..., None] > 0, acc, 0.0) * f[..., None]).sum(-2) / (ml[..., 1] * f).sum(-1, keepdim=True)
    torch.testing.assert_close(merged.view(n, -1), out.float(), rtol=2 ** -7, atol=1e-6)      # row r of scratch is request r; results are bfloat16
    with pytest.raises(K.KernelArgumentError, match="by request"):
        attend(False, work)


def test_where_one_launch_stands_for_two():
    from types import SimpleNamespace

    from jax_vllm_amd.parts.attention_backend import token_pays

    def pays(nq, nkv, n, keys, window=None, chunk=None):
        return token_pays(SimpleNamespace(nq=nq, nkv=nkv, window=window, chunk=chunk), SimpleNamespace(num_tokens=n, max_kv_len=keys))

    assert all(pays(g * kv, kv, n, keys) for g in (1, 4, 6) for kv in (1, 8) for n in (1, 64, 255) for keys in (16, 4096))
    assert not any(pays(g, 1, n, keys) for g in (7, 8, 16, 64) for n in (1, 64, 512) for keys in (16, 4096))
    # many blocks of few keys, also where a window keeps them few
    assert not pays(32, 8, 256, 512) and pays(32, 8, 256, 1024) and not pays(32, 8, 256, 4096, window=512) and not pays(32, 32, 64, 4096, chunk=256)


@pytest.mark.gpu
@pytest.mark.parametrize("n_parts,splits", [(1, 1), (2, 8), (4, 1), (4, 3)])
def test_rows_whose_scale_is_still_to_be_applied(n_parts, splits):
    """Parts of rows before their RMSNorm's scale (``UnscaledParts``, a share of the sum of squares for every part) as parts of rows behind it, and
    against the formulas: without head norms, so that the scale is in every score and every value."""
    from jax_vllm_amd.ops import kernels as K

    n, nq, nkv, ps, width, eps = 3, 12, 4, 16, 1000, 1e-5
    g = torch.Generator().manual_seed(n_parts + splits)
    contexts = [70, 1, 200]
    parts = torch.randn(n_parts, n, (nq + 2 * nkv) * D, generator=g)
    ssq = torch.rand(n, 16, generator=g) * width                    # shares behind the parts' number are not read into the scale
    ssq[:, n_parts:] = float("nan")
    scale = torch.rsqrt(ssq[:, :n_parts].double().sum(-1, keepdim=True) / width + eps)
    kp, vp = (torch.randn(1 + 13 * n, nkv, *s, generator=g).to(torch.bfloat16) for s in ((ps, D), (D, ps)))
    tables = (1 + torch.arange(13 * n, dtype=torch.int32)).view(n, 13)
    slots = torch.tensor([int(tables[i, c // ps]) * ps + c % ps for i, c in enumerate(contexts)], dtype=torch.int32).cuda()
    pos = torch.tensor(contexts, dtype=torch.int32).cuda()
    scratch = torch.empty(max(1, K.attn_decode_scratch_floats(n, nq, splits, D))).cuda()

    def attend(qkv):
        k, v, out = kp.cuda(), vp.cuda(), torch.full((n, nq * D), float("nan"), dtype=torch.bfloat16).cuda()
        K.attn_decode_token(out, qkv, slots, None, None, 0.0, None, 0, k, v, tables.cuda(), pos, nq, nkv, D, 1 / math.sqrt(D), 0, splits, scratch)
        return out.float().cpu(), k.cpu(), v.cpu()

    out, k_out, v_out = attend(K.UnscaledParts(parts.cuda(), ssq.cuda(), width, eps))
    x = (parts.double().sum(0) * scale).view(n, nq + 2 * nkv, D)
    q, k, v = (part.to(torch.bfloat16).double() for part in x.split([nq, nkv, nkv], 1))
    want = torch.zeros(n, nq, D, dtype=torch.float64)
    for i, c in enumerate(contexts):
        at = [(int(tables[i, j // ps]), j % ps) for j in range(c)]
        for h in range(nq):
            m = h // (nq // nkv)
            keys = torch.stack([kp[p, m, s].double() for p, s in at] + [k[i, m]])
            vals = torch.stack([vp[p, m, :, s].double() for p, s in at] + [v[i, m]])
            want[i, h] = torch.softmax(keys @ q[i, h] / math.sqrt(D), 0) @ vals
    torch.testing.assert_close(out.double(), want.view(n, -1), rtol=2e-2, atol=2e-2)      # as in the test above
    for i, c in enumerate(contexts):      # heads are bfloat16 once they are scaled
        torch.testing.assert_close(k_out[tables[i, c // ps], :, c % ps].double(), k[i], rtol=2 ** -7, atol=1e-6)
        torch.testing.assert_close(v_out[tables[i, c // ps], :, :, c % ps].double(), v[i], rtol=2 ** -7, atol=1e-6)
    # the scale in float before or behind the sum: a unit of a rounding of prepared heads, weights and results
    torch.testing.assert_close(out, attend((parts * scale.float()).cuda())[0], rtol=2e-2, atol=2e-2)
