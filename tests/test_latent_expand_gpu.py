"""Prompts through latent attention with every head's keys and values written out: the pages against float64 at the ends of pages, and the
whole mixer against the same step in the latent's own space over its options."""
import pytest
import torch

from .test_kernels_gpu import K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,dim,rot,vdim,rank,page_size", [(3, 64, 32, 64, 224, 16), (1, 16, 16, 32, 64, 8), (2, 32, 0, 16, 288, 24), (2, 112, 16, 128, 480, 64)])
@pytest.mark.parametrize("lens", [[1, 63], [64, 65], [130, 2, 64]], ids=str)
def test_pages(heads, dim, rot, vdim, rank, page_size, lens):
    n, d, e = sum(lens), dim + rot, rank + rot
    g = torch.Generator().manual_seed(n + e)
    count = -(-2 * n // page_size)
    pages = torch.full((count, 1, page_size, e), float("nan")).bfloat16()      # slots that nobody wrote
    slots = torch.randperm(count * page_size, generator=g)[:n]
    x = torch.randn(n, e, generator=g).bfloat16()
    pages.view(-1, e)[slots] = x
    k_up, v_up = (torch.randn(heads, r, rank, generator=g).mul(rank ** -0.5).bfloat16() for r in (dim, vdim))
    plan = K().latent_expand_plan(lens, "cuda")
    k, v = (t.cpu() for t in K().latent_expand(pages.cuda(), slots.int().cuda(), plan, k_up.view(-1, rank).cuda(), v_up.cuda(), heads, dim, rot, vdim, rank))
    tables, at = plan[2].cpu(), 0
    # one rounding to bfloat16 of a float sum
    close = lambda a, b, w: ((a.double() - b).abs() <= 2.0 ** -8 * b.abs() + rank * 2.0 ** -24 * w).all()
    for r, ln in enumerate(lens):
        for t in range(0, -(-ln // 64) * 64):
            page, off = int(tables[r, t // 64]), t % 64
            if t >= ln:
                assert (k[page, :, off] == 0).all() and (v[page, :, :, off] == 0).all()
                continue
            c = x[at + t, :rank].double()
            assert close(k[page, :, off, :dim], k_up.double() @ c, k_up.double().abs() @ c.abs())
            assert torch.equal(k[page, :, off, dim:], x[at + t, rank:].expand(heads, rot))
            assert close(v[page, :, :vdim, off], v_up.double() @ c, v_up.double().abs() @ c.abs()) and (v[page, :, vdim:, off] == 0).all()
        at += ln


@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("heads,dim,rot,rot_dims,extra", [(3, 16, 16, 16, 0), (2, 64, 32, 20, 8), (5, 24, 8, 2, 3)])
def test_queries_turn_in_place(heads, dim, rot, rot_dims, extra, interleaved):
    g = torch.Generator().manual_seed(rot_dims)
    q, ang = torch.randn(7, heads * (dim + rot) + extra, generator=g).bfloat16(), torch.randn(7, rot_dims // 2, generator=g)
    table = torch.cat([ang.cos(), ang.sin()], -1)
    got = q.cuda()
    K().latent_turn_queries(got, heads, dim, rot, rot_dims, table.cuda(), interleaved)
    want = q.double().clone()
    y = want[:, :heads * (dim + rot)].view(7, heads, -1)[:, :, dim:dim + rot_dims]
    a, b = (y[..., 0::2], y[..., 1::2]) if interleaved else y.split(rot_dims // 2, -1)
    u, w, c, s = a.clone(), b.clone(), ang.cos().double()[:, None], ang.sin().double()[:, None]
    a.copy_(u * c - w * s), b.copy_(w * c + u * s)
    assert ((got.cpu().double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -20).all()


@pytest.mark.parametrize("heads,vdim,d,gates,off", [(3, 16, 32, 1, 0), (2, 64, 96, 64, 0), (2, 64, 96, 64, 3), (5, 8, 64, 0, 0)])
def test_heads_are_cut_and_gated(heads, vdim, d, gates, off):
    g = torch.Generator().manual_seed(d)
    att, wide = torch.randn(9, heads * d, generator=g).bfloat16(), torch.randn(9, 16 + heads * max(gates, 1), generator=g).bfloat16()
    gate = wide.cuda()[:, off:off + heads * gates] if gates else None
    got = K().latent_cut_heads(att.cuda(), heads, vdim, d, gate)
    want = att.double().view(9, heads, d)[:, :, :vdim]
    if gates:
        want = want * torch.sigmoid(wide[:, off:off + heads * gates].double()).view(9, heads, gates)
    assert ((got.cpu().double() - want.reshape(9, -1)).abs() <= 2.0 ** -8 * want.reshape(9, -1).abs() + 1e-6).all()


@pytest.mark.parametrize("window,sinks,gate,q_rank,interleaved", [(None, False, "element", 24, False), (40, True, "head", 0, True), (None, True, None, 24, False), (1, False, "head", 24, False)])
@pytest.mark.parametrize("lens", [[70], [1, 64, 129, 3]], ids=str)
@pytest.mark.parametrize("page_size", [8, 24])
def test_the_mixer_both_ways(monkeypatch, window, sinks, gate, q_rank, interleaved, lens, page_size):
    from jax_vllm_amd.parts.latent_attention import LatentAttention
    from jax_vllm_amd.parts.spec import LayerMemory, PartSpec, StepContext

    heads, dim, rot, vdim, rank, hidden, n = 4, 48, 16, 32, 128, 64, sum(lens)
    part = LatentAttention(hidden, heads, dim, rot, vdim, q_rank, rank, 0.1, 1e-5, PartSpec("rotary", dict(head_dim=rot, theta=1e4, interleaved=interleaved)),
                           window, gate, sinks)
    g = torch.Generator().manual_seed(n)
    tensors = {}
    for name, t in part.tensors().items():
        x = torch.randn(t.shape, generator=g)
        tensors[name] = (x * t.shape[-1] ** -0.5).bfloat16().cuda() if t.role == "matrix" else (1 + 0.1 * x).cuda()
    part.bind(tensors, torch.bfloat16)
    per = [-(-ln // page_size) for ln in lens]
    tables, slots, positions, first = torch.zeros(len(lens), max(per), dtype=torch.int32), [], [], 1
    for r, (ln, p) in enumerate(zip(lens, per)):
        tables[r, :p] = torch.arange(first, first + p)
        slots += range(first * page_size, first * page_size + ln)
        positions += range(ln)
        first += p
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    e, x = rank + rot, torch.randn(n, hidden, generator=g).bfloat16().cuda()
    results = []
    for least in (1, 10 ** 9):
        monkeypatch.setattr(K(), "LATENT_EXPAND_MIN_TOKENS", least)
        ctx = StepContext(num_tokens=n, num_requests=len(lens), positions=i32(positions), token_req=i32(sum(([r] * ln for r, ln in enumerate(lens)), [])),
                          cu_seqlens=i32([0] + lens).cumsum(0).int(), context_lens=i32([0] * len(lens)), slot_ids=i32([0] * len(lens)), block_tables=[tables.cuda()],
                          slot_mappings=[i32(slots)], page_size=page_size, q_lens_host=lens, context_lens_host=[0] * len(lens), slot_ids_host=[0] * len(lens),
                          max_q_len=max(lens), max_kv_len=max(lens))
        pages = {"k": torch.zeros(first, 1, page_size, e, dtype=torch.bfloat16, device="cuda"), "v": torch.zeros(first, 1, e, page_size, dtype=torch.bfloat16, device="cuda")}
        assert part._written_out(x, ctx) == (least == 1)
        y = part.forward(x, ctx, LayerMemory(pages=pages, group=0))
        results.append(y.float().sum(0) if y.dim() == 3 else y.float())
    a, b = results
    # half a dozen roundings to bfloat16 each way, 2^-9 each at most, that meet in sums of dozens of terms
    assert torch.isfinite(a).all() and (a - b).norm() <= 2.0 ** -9 * 6 * b.norm()
