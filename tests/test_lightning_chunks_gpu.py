"""Linear attention by chunks of 64 tokens on the matrix unit: the ends of chunks and of their tiles of 32, more chunks than the scan
asks for at once, pieces of rows that begin off four elements, values that are not finite."""
import pytest
import torch


def run(proj, offs, lens, decay, heads, dim, vdim, state0):
    from jax_vllm_amd.ops import kernels as K

    state = state0.cuda().clone()
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    slots = torch.arange(len(lens), dtype=torch.int32, device="cuda")
    out = K.lightning_attention(proj.cuda(), *offs, state, slots, cu, decay.cuda(), heads, dim, vdim, K.lightning_chunk_plan(lens, "cuda"))
    return out.cpu().view(-1, heads, vdim), state.cpu()


def reference(q, k, v, lens, decay, state0):
    out, state, t = [], state0.double().clone(), 0
    for r, ln in enumerate(lens):
        for _ in range(ln):
            state[r] = decay.double()[:, None, None] * state[r] + k[t][:, :, None] * v[t][:, None, :]
            out.append((q[t][:, :, None] * state[r]).sum(1))
            t += 1
    return torch.stack(out), state


def numbers(n, heads, dim, vdim, dtype, pad, seed):
    g = torch.Generator().manual_seed(seed)
    proj = (torch.randn(n, pad + heads * (2 * dim + vdim), generator=g) * 0.7).to(dtype)
    act = torch.nn.functional.silu(proj.double())
    parts = act[:, pad:].split([heads * dim, heads * dim, heads * vdim], -1)
    return proj, [p.reshape(n, heads, -1) for p in parts], (pad, pad + heads * dim, pad + 2 * heads * dim)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("heads,dim,vdim,pad", [(2, 128, 128, 0), (1, 36, 160, 4), (2, 64, 33, 3)])
@pytest.mark.parametrize("lens", [[31, 32, 33], [63, 64, 65], [1, 640], [580, 129]], ids=str)
def test_ends_of_chunks(dtype, heads, dim, vdim, pad, lens):
    n = sum(lens)
    proj, (q, k, v), offs = numbers(n, heads, dim, vdim, dtype, pad, dim + n)
    decay = torch.tensor([0.97, 0.9999][:heads])
    state0 = torch.randn(len(lens), heads, dim, vdim, generator=torch.Generator().manual_seed(1)) * 0.5
    want, want_state = reference(q, k, v, lens, decay, state0)
    out, state = run(proj, offs, lens, decay, heads, dim, vdim, state0)
    # sums of up to 640 tokens and 128 keys in float: 2^-24 of some hundred steps of the largest
    assert float((out.double() - want).abs().max()) <= 2e-5 * float(want.abs().max())
    assert float((state.double() - want_state).abs().max()) <= 2e-5 * float(want_state.abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [5, 40, 70])
def test_a_value_that_is_not_finite_reaches_no_token_before_it(bad):
    heads, dim, vdim, lens = 1, 64, 96, [100]
    proj, (q, k, v), offs = numbers(100, heads, dim, vdim, torch.float32, 0, bad)
    decay, state0 = torch.tensor([0.9]), torch.zeros(1, heads, dim, vdim)
    clean, _ = run(proj, offs, lens, decay, heads, dim, vdim, state0)
    proj[bad, offs[2] + 7], proj[bad, offs[2] + 50] = float("nan"), float("inf")
    out, state = run(proj, offs, lens, decay, heads, dim, vdim, state0)
    fine = torch.ones(vdim, dtype=torch.bool)
    fine[[7, 50]] = False
    torch.testing.assert_close(out[:bad], clean[:bad], rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(out[bad:, :, fine], clean[bad:, :, fine], rtol=1e-5, atol=1e-5)
    assert not out[bad:, :, ~fine].isfinite().any() and not state[0, :, :, ~fine].isfinite().any()
