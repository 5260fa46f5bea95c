"""One token of the gated delta rule and of gated linear attention in one launch, against float64: heads that fill a block and heads that
leave most of it idle, every length of filter, requests without a token, columns that begin anywhere in a wider row."""
import pytest
import torch
from torch.nn.functional import silu, softplus

from .test_kernels_gpu import K

pytestmark = pytest.mark.gpu
SIZES = [(128, 128), (127, 124), (1, 4), (36, 20), (128, 4), (17, 128), (65, 64)]


def steps_of(lens):
    cu = torch.tensor([0] + lens).cumsum(0).int()
    slots = torch.randperm(len(lens) + 2, generator=torch.Generator().manual_seed(1))[:len(lens)].int()
    return cu, slots


def gated_norm(o, norm, gate, eps, scale):
    o = o / torch.sqrt((o * o).mean(-1, keepdim=True) + eps)
    return o * norm.double() * silu(gate) * scale


def check(got, want, limit, dtype):
    # sums of up to 128 float terms and a dozen roundings before them: 150 * 2^-24 of the terms' magnitudes, which a result
    # of root mean square 1 that many terms cancel in can show 15 times over; then the result's own rounding
    own = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -24
    assert torch.isfinite(got).all()
    assert ((got.double() - want).abs() <= own * want.abs() + 150 * 2.0 ** -24 * 15 * limit).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("dim,vdim", SIZES)
@pytest.mark.parametrize("taps,at,lens", [(4, 0, [1, 1, 1]), (1, 3, [1, 0, 1, 1]), (2, 8, [1]), (8, 1, [0, 1, 1, 1, 0])], ids=str)
def test_delta(dtype, dim, vdim, taps, at, lens):
    g = torch.Generator().manual_seed(dim * 131 + vdim + taps)
    heads, n = 3, sum(lens)
    qk, inner = heads * dim, heads * vdim
    cu, slots = steps_of(lens)
    proj = torch.randn(n, at + 2 * qk + 2 * inner + 2 * heads + 5, generator=g).to(dtype)
    channels = 2 * qk + inner
    conv_w = torch.randn(channels, taps, generator=g) * 0.5
    conv0 = torch.randn(len(lens) + 2, taps - 1, channels, generator=g)
    s0 = torch.randn(len(lens) + 2, heads, dim, vdim, generator=g)
    dt, a_log, norm = torch.randn(heads, generator=g), torch.randn(heads, generator=g) - 2, 1 + 0.1 * torch.randn(vdim, generator=g)
    conv, s = conv0.cuda(), s0.cuda()
    assert K().recurrence_token_possible(dim, vdim, s)
    got = K().delta_token(proj.cuda(), at, conv_w.cuda(), conv, dt.cuda(), a_log.cuda(), 1e-6, dim ** -0.5, norm.cuda(), 1e-5, 0.5, s,
                          slots.cuda(), cu.cuda(), heads, dim, vdim)
    conv_want, s_want, t = conv0.clone(), s0.double(), 0
    for r, ln in enumerate(lens):
        if not ln:
            continue
        x, slot = proj[t].double()[at:], int(slots[r])
        window = torch.cat([conv0[slot].double(), x[None, :channels]])
        conv_want[slot] = window[1:].float()
        y = silu((window * conv_w.double().T).sum(0))
        q, k, v = y[:qk].view(heads, dim), y[qk:2 * qk].view(heads, dim), y[2 * qk:].view(heads, vdim)
        q, k = (z / torch.sqrt((z * z).sum(-1, keepdim=True) + 1e-6) for z in (q, k))
        gate, (raw, beta) = x[channels:channels + inner].view(heads, vdim), x[channels + inner:channels + inner + 2 * heads].view(2, heads)
        fade = torch.exp(-torch.exp(a_log.double()) * softplus(raw + dt.double(), threshold=1e9))
        old = s_want[slot] * fade[:, None, None]
        u = torch.sigmoid(beta)[:, None] * (v - (k[:, :, None] * old).sum(1))
        s_want[slot] = old + k[:, :, None] * u[:, None, :]
        o = (q[:, :, None] * s_want[slot]).sum(1) * dim ** -0.5
        want = gated_norm(o, norm, gate, 1e-5, 0.5)
        check(got[t].cpu(), want.reshape(-1), ((norm.double() * silu(gate)).abs() + 0.1).reshape(-1) * dim ** 0.5, dtype)
        t += 1
    assert torch.equal(conv.cpu(), conv_want)
    # the state's own terms: a prediction of dim terms of size 1, a decay by the exponential of a float
    assert ((s.cpu().double() - s_want).abs() <= 2.0 ** -24 * (dim + 40) * (2 + s_want.abs())).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("dim,vdim", SIZES)
@pytest.mark.parametrize("rank,at,lens", [(16, 0, [1, 1, 1]), (1, 3, [1, 0, 1]), (64, 8, [1]), (13, 0, [0, 1, 1, 0])], ids=str)
def test_gated_linear(dtype, dim, vdim, rank, at, lens):
    g = torch.Generator().manual_seed(dim * 131 + vdim + rank)
    heads, n = 2, sum(lens)
    qk, inner = heads * dim, heads * vdim
    cu, slots = steps_of(lens)
    proj = torch.randn(n, at + 2 * qk + 2 * inner + rank + 3, generator=g).to(dtype)
    up, bias = (torch.randn(qk, rank, generator=g) * rank ** -0.5).to(dtype), 2 + torch.randn(qk, generator=g)
    s0 = torch.randn(len(lens) + 2, heads, dim, vdim, generator=g)
    norm, s = 1 + 0.1 * torch.randn(vdim, generator=g), s0.cuda()
    assert K().gated_linear_token_possible(dim, vdim, rank, s)
    got = K().gated_linear_token(proj.cuda(), at, up.cuda(), bias.cuda(), 16.0, dim ** -0.5, norm.cuda(), 1e-5, s, slots.cuda(), cu.cuda(),
                                 heads, dim, vdim)
    s_want, t = s0.double(), 0
    for r, ln in enumerate(lens):
        if not ln:
            continue
        x, slot = proj[t].double()[at:], int(slots[r])
        q, k, v = x[:qk].view(heads, dim), x[qk:2 * qk].view(heads, dim), x[2 * qk:2 * qk + inner].view(heads, vdim)
        gate, low = x[2 * qk + inner:2 * qk + 2 * inner].view(heads, vdim), x[2 * qk + 2 * inner:2 * qk + 2 * inner + rank]
        z = up.double() @ low + bias.double()
        fade = torch.sigmoid(z) ** (1 / 16.0)
        s_want[slot] = fade.view(heads, dim, 1) * s_want[slot] + k[:, :, None] * v[:, None, :]
        o = (q[:, :, None] * s_want[slot]).sum(1) * dim ** -0.5
        want = gated_norm(o, norm, gate, 1e-5, 1.0)
        check(got[t].cpu(), want.reshape(-1), ((norm.double() * silu(gate)).abs() + 0.1).reshape(-1) * dim ** 0.5, dtype)
        t += 1
    assert ((s.cpu().double() - s_want).abs() <= 2.0 ** -24 * (rank + 40) * (4 + s_want.abs())).all()


def test_what_the_launch_does_not_take():
    s = torch.zeros(1, 1, 128, 132, device="cuda")
    assert not K().recurrence_token_possible(129, 128, s) and not K().recurrence_token_possible(128, 132, s)
    assert not K().recurrence_token_possible(128, 6, s) and not K().recurrence_token_possible(8, 8, s.view(-1)[1:])
    assert not K().gated_linear_token_possible(8, 8, 65, s)
