"""Heads of many tokens into their pages by one launch: slots that run on, begin inside a page, stand alone, or are not stored."""
import pytest
import torch

from .test_kernels_gpu import DTYPES, K, randn, rope_reference, tol


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,d,ps,n", [(32, 8, 128, 16, 256), (3, 1, 128, 8, 257), (6, 3, 64, 24, 271), (4, 2, 256, 16, 300), (5, 5, 48, 8, 290)])
def test_many_tokens_into_their_pages(dtype, nq, nkv, d, ps, n):
    pages, eps = n // ps + 70, 1e-6
    qkv = randn(n, (nq + 2 * nkv) * d, dtype=dtype, seed=n)
    # single tokens, a run from inside a page, tokens that are not stored, a run to the end that begins off a multiple of 8
    slots = [(3 + 2 * i) * ps + i % ps for i in range(19)]
    at = 45 * ps + 3
    slots += list(range(at, at + 101)) + [-1] * 5
    at = (45 + 101 // ps + 3) * ps + (0 if ps == 24 else 5)
    slots += list(range(at, at + n - len(slots)))
    assert len(slots) == n and max(slots) < pages * ps and len(set(s for s in slots if s >= 0)) == n - 5
    s = torch.tensor(slots, dtype=torch.int32).cuda()
    pos = torch.arange(n, dtype=torch.int32).cuda()
    freq = (1.0 / (1e4 ** (torch.arange(0, d, 2, dtype=torch.float32) / d))).cuda()
    qw, kw = 1 + 0.1 * randn(d, seed=1), 1 + 0.1 * randn(d, seed=2)
    kp, vp = torch.zeros(pages, nkv, ps, d, dtype=dtype).cuda(), torch.zeros(pages, nkv, d, ps, dtype=dtype).cuda()
    x = qkv.float().view(n, -1, d).clone()
    K().qk_norm_rope_write(qkv, s, qw, kw, eps, K().rope_table(pos, freq), d, False, kp, vp, ps, nq, nkv, d)
    norm = lambda t, w: t * torch.rsqrt((t * t).mean(-1, keepdim=True) + eps) * w
    q = rope_reference(norm(x[:, :nq], qw), pos, freq, d, False)
    k = rope_reference(norm(x[:, nq:nq + nkv], kw), pos, freq, d, False)
    want_k, want_v = torch.zeros(pages, nkv, ps, d).cuda(), torch.zeros(pages, nkv, d, ps).cuda()
    for i, c in enumerate(slots):
        if c >= 0:
            want_k[c // ps, :, c % ps] = k[i]
            want_v[c // ps, :, :, c % ps] = x[i, nq + nkv:]
    close = tol(dtype, f32=2e-5, bf16=2e-2)
    torch.testing.assert_close(qkv.float().view(n, -1, d)[:, :nq], q, **close)
    torch.testing.assert_close(kp.float(), want_k, **close)
    assert torch.equal(vp.float(), want_v)
