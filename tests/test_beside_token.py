"""The heads of an attention prepared beside a recurrent mixer's token, in one launch: the bits of two launches, with waves and blocks that have
no head, requests without a token, and sizes whose heads go through another kernel."""
import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("kind", ["delta", "gated"])
@pytest.mark.parametrize("n,nq,nkv,dk,heads,dim,empty", [(1, 4, 2, 128, 2, 128, 0), (16, 16, 4, 128, 16, 128, 0), (5, 3, 1, 72, 3, 40, 2),
                                                         (130, 4, 2, 64, 2, 64, 0), (3, 1, 1, 800, 1, 16, 0)])
def test_the_bits_of_two_launches(n, nq, nkv, dk, heads, dim, empty, kind, dtype):
    from jax_vllm_amd.ops import kernels as K

    g = torch.Generator().manual_seed(n + dk)
    page, right_at, rank, requests = 16, (nq + 2 * nkv) * dk, 8, n + empty
    width = right_at + heads * 4 * dim + max(2 * heads, rank)
    proj = torch.randn(n, width + 7, generator=g).to(dtype).cuda()
    rot = dk // 4 * 2
    cos_sin = torch.randn(n, rot, generator=g).cuda()
    slots = torch.randperm(4 * page * (n // page + 1), generator=g)[:n].int().cuda()
    shape = (4 * (n // page + 1), nkv, page, dk)
    # the requests without a token come last
    cu = torch.tensor(list(range(n + 1)) + [n] * empty, dtype=torch.int32).cuda()
    slot_ids = torch.randperm(requests, generator=g).int().cuda()
    norm = torch.rand(dim, generator=g).cuda()
    state = torch.randn(requests, heads, dim, dim, generator=g).cuda()
    conv_w, conv = torch.randn(3 * heads * dim, 4, generator=g).cuda(), torch.randn(requests, 3, 3 * heads * dim, generator=g).cuda()
    bias, a_log = torch.randn(heads, generator=g).cuda(), torch.randn(heads, generator=g).cuda()
    up, up_bias = torch.randn(heads * dim, rank, generator=g).to(dtype).cuda(), torch.randn(heads * dim, generator=g).cuda()

    def run(beside):
        k, v = torch.zeros(shape, dtype=dtype, device="cuda"), torch.zeros((shape[0], nkv, dk, page), dtype=dtype, device="cuda")
        s, c = state.clone(), conv.clone()
        held = K.HeldToken() if beside else None
        if kind == "delta":
            y = K.delta_token(proj, right_at, conv_w, c, bias, a_log, 1e-6, dim ** -0.5, norm, 1e-5, 1.0, s, slot_ids, cu, heads, dim, dim, hold=held)
        else:
            y = K.gated_linear_token(proj, right_at, up, up_bias, 16.0, dim ** -0.5, norm, 1e-5, s, slot_ids, cu, heads, dim, dim, hold=held)
        q = K.attn_prepare_wide(proj, None, None, None, 0.0, cos_sin, rot, slots, k, v, page, nq, nkv, dk, dk, dk, norm_per_head=True, beside=held)
        return q, k, v, s, c, held.out if beside else y

    for a, b in zip(run(False), run(True)):
        assert torch.equal(a, b)


def test_a_launch_that_nobody_took_is_no_result():
    from types import SimpleNamespace

    from jax_vllm_amd.ops import kernels as K
    from jax_vllm_amd.parts.recurrent import GatedDeltaMixer, GatedLinearAttention

    held = object.__new__(K.HeldToken)
    held.out, held.taken = torch.zeros(1, 4), False
    for mixer in (GatedDeltaMixer, GatedLinearAttention):
        with pytest.raises(K.KernelArgumentError, match="not taken"):
            mixer.finish_token(SimpleNamespace(w_o=torch.zeros(4, 4)), held)
    held.taken = True
    assert held.result() is held.out


@pytest.mark.gpu
def test_a_launch_is_taken_once():
    from jax_vllm_amd.ops import kernels as K

    heads, dim = 2, 64
    proj = torch.randn(2, 3 * 64 + heads * 4 * dim + 8, device="cuda")
    cu, slots = torch.arange(3, dtype=torch.int32, device="cuda"), torch.arange(2, dtype=torch.int32, device="cuda")
    state = torch.zeros(2, heads, dim, dim, device="cuda")
    up, held = torch.zeros(heads * dim, 8, device="cuda"), K.HeldToken()
    K.gated_linear_token(proj, 3 * 64, up, torch.zeros(heads * dim, device="cuda"), 16.0, 1.0, torch.ones(dim, device="cuda"), 1e-5, state, slots, cu, heads, dim,
                         dim, hold=held)
    with pytest.raises(K.KernelArgumentError, match="not taken"):
        held.result()
    prepare = lambda: K.attn_prepare_wide(proj, None, None, None, 0.0, None, 0, None, None, None, 16, 1, 1, 64, 64, 64, beside=held)
    prepare()
    assert held.result() is held.out and held.out.isfinite().all()
    with pytest.raises(K.KernelArgumentError, match="before"):
        prepare()
