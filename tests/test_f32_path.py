"""The 32-bit path's products and attention on the matrix cores: against float64, at the edges of tiles and parts, and the
products bit by bit across batches."""
import pytest
import torch

from .test_kernels_gpu import K, build_paged, randn


# ------------------------------------------------------------------ matrix products
@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 15, 16, 17, 32, 33, 63, 65, 127, 129])
@pytest.mark.parametrize("n,k", [(1, 1), (15, 127), (16, 128), (33, 129), (63, 2047), (4099, 516), (8200, 144)])
def test_gemm_f32_tiles_and_parts(m, n, k):
    a, w = randn(m, k, seed=m), randn(n, k, seed=n + k)
    out = K().gemm_f32(a, w)
    want = a.double() @ w.double().T
    # eight chains of at most k / 8 + 16 fused steps and eight sums: far inside the bound of one chain of k
    assert ((out.double() - want).abs() <= 2.0 ** -24 * (k / 8 + 24) * (a.double().abs() @ w.double().abs().T)).all()
    # whatever tile the batch takes, a row's bits are the same
    for rows in (slice(0, 1), slice(m // 2, m // 2 + 1), slice(0, (m + 1) // 2)):
        assert torch.equal(K().gemm_f32(a[rows].contiguous(), w), out[rows])


# ------------------------------------------------------------------ attention
def reference(q, k, v, pos, scale, window, chunk, keep, cap, sinks):
    g = q.shape[1] // k.shape[1]
    kk, vv = (torch.repeat_interleave(x.double(), g, dim=1) for x in (k, v))
    s = torch.einsum("qhd,khd->hqk", q.double(), kk) * scale
    if cap:
        s = cap * torch.tanh(s / cap)
    i, j = pos[:, None], torch.arange(k.shape[0])[None, :]
    seen = j <= i
    if window:
        seen &= (i - j < window) | (j < keep)
    if chunk:
        seen &= (i // chunk == j // chunk) | (j < keep)
    s = s.masked_fill(~seen[None], float("-inf"))
    if sinks is not None:
        s = torch.cat([s, sinks.double()[:, None, None].expand(-1, s.shape[1], 1)], -1)
    p = torch.softmax(s, -1)[..., :k.shape[0]]
    return torch.einsum("hqk,khd->qhd", p, vv)


# nq, nkv, d, page size, [(cached, new)], window, chunk, keep, cap, sinks
CASES = [
    (4, 2, 32, 4, [(0, 1), (0, 5), (14, 3), (15, 1), (16, 1)], None, None, 0, 0.0, False),
    (8, 2, 64, 8, [(0, 33), (31, 2), (200, 1)], None, None, 0, 0.0, True),
    (6, 2, 96, 16, [(300, 1), (0, 17), (7, 50)], 24, None, 5, 0.0, True),
    (16, 4, 128, 16, [(205, 1), (0, 70), (1000, 9)], None, None, 0, 50.0, False),
    (16, 4, 128, 16, [(205, 1), (409, 1), (614, 1)], 64, None, 16, 30.0, True),
    (8, 2, 128, 32, [(0, 130), (90, 40)], None, 48, 0, 0.0, True),
    (8, 2, 128, 16, [(0, 130), (90, 40)], None, 48, 20, 0.0, False),
    (16, 1, 256, 16, [(10, 3), (255, 1), (0, 40)], 100, None, 0, 0.0, True),
    (40, 2, 64, 16, [(37, 1), (0, 9)], None, None, 0, 0.0, False),                  # more than 16 rows for one token
]


def paged(case, seed=3):
    nq, nkv, d, page, reqs = case[:5]
    g = torch.Generator().manual_seed(seed)
    ks, vs = ([torch.randn(c + n, nkv, d, generator=g) for c, n in reqs] for _ in range(2))
    qs = [torch.randn(n, nq, d, generator=g) for _, n in reqs]
    return ks, vs, qs, build_paged(ks, vs, page)


def run_kernel(case, qs, k_pages, v_pages, tables, sinks, splits=1):
    from jax_vllm_amd.parts.attention_backend import f32_work_items

    nq, nkv, d, _, reqs, window, chunk, keep, cap, _ = case
    lens, ctx = [n for _, n in reqs], [c for c, _ in reqs]
    items = f32_work_items(lens, ctx, nq // nkv, K().attn_f32_rows())
    total, stride = sum(lens), (nq + 2 * nkv) * d
    buf = torch.zeros(total, stride)
    buf[:, :nq * d] = torch.cat(qs).reshape(total, nq * d)
    cu = torch.tensor([0] + lens).cumsum(0).int()
    out = torch.full((total, nq * d), float("nan")).cuda()
    K().attn_f32(out, buf.cuda(), stride, k_pages.cuda(), v_pages.cuda(), tables.cuda(), cu.cuda(), torch.tensor(ctx).int().cuda(),
                 torch.tensor(items).int().cuda(), len(items), nq, nkv, d, d ** -0.5, K().key_window(window, chunk), splits,
                 torch.full((K().attn_f32_part_floats(len(items), nkv, splits, d),), float("nan")).cuda(), sinks=None if sinks is None else sinks.cuda(), cap=cap, keep=keep)
    return out.cpu().view(total, nq, d)


@pytest.mark.gpu
@pytest.mark.parametrize("splits", [1, 2, 9])          # 9: blocks without a key among them
@pytest.mark.parametrize("case", CASES, ids=[f"h{c[0]}g{c[1]}d{c[2]}p{c[3]}w{c[5]}c{c[6]}k{c[7]}" for c in CASES])
def test_attention_f32(case, splits):
    nq, nkv, d, _, reqs, window, chunk, keep, cap, with_sinks = case
    ks, vs, qs, (k_pages, v_pages, tables) = paged(case)
    sinks = torch.linspace(-1.0, 2.0, nq) if with_sinks else None
    out = run_kernel(case, qs, k_pages, v_pages, tables, sinks, splits)
    want = torch.cat([reference(q, k, v, torch.arange(c, c + n), d ** -0.5, window, chunk, keep, cap, sinks)
                      for q, k, v, (c, n) in zip(qs, ks, vs, reqs)])
    # sums over d and over the keys in float, the scores' error enters the exponent: a few 2^-24 sqrt(d) of scores up to ~5
    torch.testing.assert_close(out.double(), want, rtol=1e-5, atol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("d,page", [(32, 4), (128, 16)])
def test_a_value_that_is_not_finite_stays_with_those_who_see_it(d, page):
    """A key in the middle of a tile holds infinity or NaN: rows before it (and rows whose window has passed it) are as if it
    were not there, and stale slots behind the last key are nobody's."""
    case = (4, 2, d, page, [(0, 40), (3, 21)], 12, None, 0, 0.0, False)
    ks, vs, qs, (k_pages, v_pages, tables) = paged(case)
    clean = run_kernel(case, qs, k_pages, v_pages, tables, None)
    bad = 21                                                            # of the first request
    k_pages, v_pages = k_pages.clone(), v_pages.clone()
    slot = int(tables[0, bad // page])
    v_pages[slot, :, :, bad % page] = float("nan")
    k_pages[slot, :, bad % page] = float("inf")
    last = int(tables[1, 23 // page])
    v_pages[last, :, :, 23 % page + 1:] = float("inf")                  # behind the second request's last key
    out = run_kernel(case, qs, k_pages, v_pages, tables, None)
    sees = torch.zeros(out.shape[0], dtype=torch.bool)
    sees[bad:bad + 12] = True
    assert torch.isnan(out[sees]).all()
    torch.testing.assert_close(out[~sees], clean[~sees], rtol=1e-6, atol=1e-6)      # one key walked by hand instead of by product


def test_f32_work_items_hold_every_row_once():
    from jax_vllm_amd.parts.attention_backend import f32_work_items

    lens, ctx, g = [1, 40, 3, 16], [900, 0, 12, 64], 3
    for rows in (16, 32):
        items = f32_work_items(lens, ctx, g, rows)
        covered = sorted((r, m) for r, m0 in items for m in range(m0, min(m0 + rows, lens[r] * g)))
        assert covered == [(r, m) for r, n in enumerate(lens) for m in range(n * g)]
        assert items[0][0] == 0                                          # the request with the most keys first


def run_step(case_sizes, reqs, pages, tables, queries, window=None, chunk=None, keep=0, cap=None, sinks=None, dtype=torch.float32, plans=None):
    """A step of these requests [(cached, new)] through the backend, with its own plan: the kernel's choice of blocks included.
    ``plans``: a list that receives the step's plan."""
    from types import SimpleNamespace

    from jax_vllm_amd.parts import attention_backend
    from jax_vllm_amd.parts.spec import LayerMemory, StepContext

    nq, nkv, d, page = case_sizes
    lens, ctx = [n for _, n in reqs], [c for c, _ in reqs]

    def i32(values):
        return torch.tensor(values, dtype=torch.int32).cuda()

    step = StepContext(num_tokens=sum(lens), num_requests=len(reqs), positions=i32([c + i for c, n in reqs for i in range(n)]),
                       token_req=i32([r for r, n in enumerate(lens) for _ in range(n)]),
                       cu_seqlens=i32([0] + torch.tensor(lens).cumsum(0).tolist()), context_lens=i32(ctx), slot_ids=i32([0] * len(reqs)),
                       block_tables=[tables.cuda()], slot_mappings=[None], page_size=page, q_lens_host=lens, context_lens_host=ctx,
                       slot_ids_host=[0] * len(reqs), max_q_len=max(lens), max_kv_len=max(c + n for c, n in reqs))
    att = SimpleNamespace(nq=nq, nkv=nkv, d=d, window=window, chunk=chunk, q_row_stride=nq * d, sinks=sinks, softcap=cap, keep_first=keep,
                          scale=d ** -0.5)
    out = torch.full((sum(lens), nq * d), float("nan"), dtype=dtype).cuda()
    attention_backend.run(att, out, torch.cat(queries).reshape(sum(lens), nq * d).to(dtype).cuda(), step,
                          LayerMemory(pages={"k": pages[0].to(dtype).cuda(), "v": pages[1].to(dtype).cuda()}, group=0))
    if plans is not None:
        plans.extend(step.plans.values())
    return out.cpu()


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [(16, 4, 128, 16), (8, 1, 256, 16), (12, 4, 32, 4), (4, 2, 64, 24)])
@pytest.mark.parametrize("mask", [{}, {"window": 300}, {"window": 40, "keep": 20}, {"window": 500, "keep": 700}, {"chunk": 384}, {"cap": 30.0}])
def test_a_token_s_bits_depend_on_what_it_sees_alone(sizes, mask):
    """The same tokens over the same keys: alone, beside other requests (few and many: an item's ranges with blocks of their own or
    in one), and cut into portions."""
    nq, nkv, d, page = sizes
    g = torch.Generator().manual_seed(d)
    total = 1100
    lengths = [total, 5, 2500] + [700] * 40
    ks, vs = ([torch.randn(n, nkv, d, generator=g) for n in lengths] for _ in range(2))
    q = [torch.randn(n, nq, d, generator=g) for n in lengths]
    *pages, tables = build_paged(ks, vs, page)

    def step(who):                                # [(request, cached, new)]
        return run_step(sizes, [(c, n) for _, c, n in who], pages, tables[[r for r, _, _ in who]], [q[r][c:c + n] for r, c, n in who], **mask)

    alone = step([(0, total - 1, 1)])
    assert torch.isfinite(alone).all()
    for others in ([(1, 4, 1)], [(r, lengths[r] - 1, 1) for r in range(1, 17)], [(r, 600, 1) for r in range(3, 43)], [(2, 0, 2500)]):
        assert torch.equal(step([(0, total - 1, 1)] + others)[:1], alone)
        assert torch.equal(step(others + [(0, total - 1, 1)])[-1:], alone)
    whole = step([(0, 0, total)])
    assert torch.equal(whole[-1:], alone)
    at = 0
    for n in (1, 250, 18, 400, 431):              # the ends of tiles and ranges inside and between portions
        assert torch.equal(step([(0, at, n)]), whole[at:at + n])
        at += n
    assert at == total


def test_the_ranges_that_a_work_item_may_touch():
    from jax_vllm_amd.parts.attention_backend import f32_ranges

    for rows in (1, 16):
        for kv_len in (1, 16, 255, 256, 257, 300, 1000, 5000):
            for window, keep in ((0, 0), (1, 0), (40, 20), (257, 0), (241, 300), (3000, 16), (-384, 0), (-7, 33)):
                bound = f32_ranges(kv_len, window, keep, rows, 256)
                for last in {kv_len - 1, max(0, kv_len - 130), max(0, kv_len - 256)}:
                    first = max(0, last - rows + 1)
                    begin = max(0, first - window + 1) if window > 0 else first - first % -window if window else 0
                    begin = begin // 16 * 16                                       # whole tiles
                    touched = {j // 256 for j in list(range(min(keep, begin))) + list(range(begin, last + 1))}
                    assert len(touched) <= bound, (kv_len, window, keep, rows, last)


@pytest.mark.gpu
def test_a_request_s_logits_do_not_depend_on_its_company():
    """A dense model in 32 bits through the engine: a prompt's portions and decoded tokens, alone and beside others, to the bit
    (steps of 256 tokens and more prepare heads by another kernel, so both walks cut alike)."""
    import numpy as np

    from jax_vllm_amd import LLM
    from jax_vllm_amd.engine.entries import StepEntry

    cfg = dict(architectures=["Qwen3ForCausalLM"], hidden_size=256, num_attention_heads=8, num_key_value_heads=2, head_dim=64,
               intermediate_size=384, vocab_size=512, num_hidden_layers=3, rope_theta=1e6, rms_norm_eps=1e-6, tie_word_embeddings=False,
               max_position_embeddings=4096)
    rng = np.random.default_rng(3)
    mine = rng.integers(0, 512, size=640).tolist()
    others = [rng.integers(0, 512, size=n).tolist() for n in (3, 900, 40, 333, 17, 600, 64, 5, 128, 450)]

    def walk(cuts, company):
        """My logits at every cut's end, with the others' prompts in the first step and their tokens in the rest."""
        llm = LLM(cfg, random_seed=5, dtype="fp32", block_size=16, num_blocks=1 + 11 * 64, max_num_seqs=11, max_model_len=1024,
                  max_num_batched_tokens=4096, enable_prefix_cache=False)
        core, out, at = llm.core, [], 0
        names = ["me"] + [f"o{i}" for i in range(len(others))] if company else ["me"]
        for name in names:
            core.start_request(name)
        for step, n in enumerate(cuts):
            entries = [StepEntry("me", mine[at:at + n], [n - 1])]
            if company:
                entries += [StepEntry(f"o{i}", t if step == 0 else [t[step % len(t)]], [0]) for i, t in enumerate(others)]
            if step % 2:
                entries = entries[::-1]                    # I am the last request of every other step
            logits = core.run(entries).cpu()
            out.append(logits[-1] if step % 2 else logits[0])
            at += n
        return torch.stack(out)

    cuts = [300, 1, 1, 20, 1, 310] + [1] * 7
    assert sum(cuts) == 640
    alone = walk(cuts, False)
    assert torch.isfinite(alone).all() and torch.equal(walk(cuts, True), alone)
