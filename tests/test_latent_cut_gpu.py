"""Latent attention in bfloat16: a prompt's error against float64 is the same whole and in portions, with the gate on float sums."""
import pytest
import torch

pytestmark = pytest.mark.gpu
HEADS, DIM, ROT, VDIM, RANK, HIDDEN, PAGE = 8, 64, 32, 64, 224, 512, 16


def layer(gate, window, g):
    from jax_vllm_amd.parts.latent_attention import LatentAttention
    from jax_vllm_amd.parts.spec import PartSpec

    part = LatentAttention(HIDDEN, HEADS, DIM, ROT, VDIM, 128, RANK, (DIM + ROT) ** -0.5, 1e-5, PartSpec("rotary", dict(head_dim=ROT, theta=1e4)), window, gate)
    tensors = {}
    for name, t in part.tensors().items():
        x = torch.randn(t.shape, generator=g)
        tensors[name] = ((x * t.shape[-1] ** -0.5).bfloat16() if t.role == "matrix" else 1.5 + 0.03 * x).cuda()
    part.bind(tensors, torch.bfloat16)
    return part, {name: t.double() for name, t in tensors.items()}


def in_portions(part, x, lens, cuts):
    """The layer's rows of requests of ``lens`` tokens, their tokens up to ``cuts`` of each in a step of their own; and the rotation's table."""
    from jax_vllm_amd.parts.spec import LayerMemory, StepContext

    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    per = [-(-ln // PAGE) for ln in lens]
    firsts = [1 + sum(per[:r]) for r in range(len(lens))]
    tables = torch.zeros(len(lens), max(per), dtype=torch.int32)
    for r, p in enumerate(per):
        tables[r, :p] = torch.arange(firsts[r], firsts[r] + p)
    e, count = RANK + ROT, 1 + sum(per)
    mem = LayerMemory(pages={"k": torch.zeros(count, 1, PAGE, e, dtype=torch.bfloat16, device="cuda"),
                             "v": torch.zeros(count, 1, e, PAGE, dtype=torch.bfloat16, device="cuda")}, group=0)
    starts, out, table = [sum(lens[:r]) for r in range(len(lens))], torch.empty(sum(lens), HIDDEN, dtype=torch.float64, device="cuda"), None
    for lo, hi in ((lambda ln: 0, lambda ln: min(cuts, ln)), (lambda ln: min(cuts, ln), lambda ln: ln)):
        own = [(r, lo(ln), hi(ln)) for r, ln in enumerate(lens) if hi(ln) > lo(ln)]
        if not own:
            continue
        rows = i32([starts[r] + t for r, a, b in own for t in range(a, b)]).long()
        q_lens, at = [b - a for _, a, b in own], [a for _, a, _ in own]
        ctx = StepContext(num_tokens=len(rows), num_requests=len(own), positions=i32([t for _, a, b in own for t in range(a, b)]),
                          token_req=i32([i for i, n in enumerate(q_lens) for _ in range(n)]), cu_seqlens=i32([0] + q_lens).cumsum(0).int(),
                          context_lens=i32(at), slot_ids=i32([0] * len(own)), block_tables=[tables[[r for r, _, _ in own]].cuda()],
                          slot_mappings=[i32([firsts[r] * PAGE + t for r, a, b in own for t in range(a, b)])], page_size=PAGE, q_lens_host=q_lens,
                          context_lens_host=at, slot_ids_host=[0] * len(own), max_q_len=max(q_lens), max_kv_len=max(b for _, _, b in own))
        y = part.forward(x[rows].contiguous(), ctx, mem).double()
        out[rows] = y.sum(0) if y.dim() == 3 else y
        if len(own) == len(lens) and cuts >= max(lens):
            table = part.position.rotation_table(ctx).double()
    return out, table


def exact(w, x, table, lens, gate, window, scale):
    norm = lambda v, weight: v / torch.sqrt((v * v).mean(-1, keepdim=True) + 1e-5) * weight
    n, half = len(x), ROT // 2

    def turn(v):
        c, s = (t.view(n, *[1] * (v.dim() - 2), half) for t in (table[:, :half], table[:, half:ROT]))
        a, b = v[..., :half], v[..., half:]
        return torch.cat([a * c - b * s, b * c + a * s], -1)

    x = x.double()
    q = (norm(x @ w["q_down.weight"].T, w["q_norm.weight"]) @ w["q_up.weight"].T).view(n, HEADS, DIM + ROT)
    q = torch.cat([q[..., :DIM], turn(q[..., DIM:])], -1)
    kv = x @ w["kv_down.weight"].T
    c, rotated = norm(kv[:, :RANK], w["kv_norm.weight"]), turn(kv[:, RANK:])
    k = torch.cat([(c @ w["k_up.weight"].T).view(n, HEADS, DIM), rotated[:, None].expand(n, HEADS, ROT)], -1)
    v, out, at = (c @ w["v_up.weight"].T).view(n, HEADS, VDIM), [], 0
    for ln in lens:
        qs, ks, vs = (t[at:at + ln].transpose(0, 1) for t in (q, k, v))
        back = torch.arange(ln, device="cuda")[:, None] - torch.arange(ln, device="cuda")
        hidden = (back < 0) | (back >= (window or ln))
        out.append((torch.softmax((qs @ ks.transpose(1, 2) * scale).masked_fill(hidden, -float("inf")), -1) @ vs).transpose(0, 1))
        at += ln
    o = torch.cat(out).reshape(n, -1)
    if gate:
        by = torch.sigmoid(x @ w["gate.weight"].T)
        o = o * (by.repeat_interleave(VDIM, 1) if gate == "head" else by)
    return o @ w["o_proj.weight"].T


@pytest.mark.parametrize("gate,window", [("element", None), ("head", 100)])
@pytest.mark.parametrize("lens,cuts", [([900], 400), ([9] * 80, 5)], ids=["one", "short"])
def test_error_does_not_depend_on_the_cut(gate, window, lens, cuts):
    g = torch.Generator().manual_seed(len(lens))
    part, w = layer(gate, window, g)
    x = torch.randn(sum(lens), HIDDEN, generator=g).bfloat16().cuda()
    whole, table = in_portions(part, x, lens, max(lens))
    cut, _ = in_portions(part, x, lens, cuts)
    want = exact(w, x, table, lens, gate, window, part.scale)
    a, b = ((y - want).norm() / want.norm() for y in (whole, cut))
    # the same roundings both ways, of more than 300,000 results: the norms of their errors agree to about 0.2 %; one more
    # rounding to bfloat16 before the gate is 4 to 8 %
    assert a <= 1.015 * b and b <= 1.015 * a and a <= 6 * 2.0 ** -9, (float(a), float(b))
