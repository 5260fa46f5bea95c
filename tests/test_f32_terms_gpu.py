"""Float rows with their terms for the next 32-bit product: the kernels that make the rows leave the bits of a launch that splits them."""
import ctypes

import pytest
import torch

from .test_kernels_gpu import K, randn


def split(x, fragments):
    """The terms of x by the launch of their own."""
    k_, (m, k) = K(), x.shape
    t = k_.f32_terms(m, k, fragments, x.device)
    lib = k_.library.core()
    fn = lib.jv_split_fragments_f32 if fragments else lib.jv_split_rows_f32
    assert fn(k_._ptr(t), k_._ptr(x), ctypes.c_int(m), ctypes.c_int(k), k_._stream()) == 0
    return t


def same(rows, fragments):
    """Bit for bit; rows behind the last one of a fragment hold anything."""
    want, got = split(rows.x, fragments), rows.terms
    if fragments:
        m, k = rows.shape
        want, got = (t.view(-1, k // 32, 3, 4, 32, 8).transpose(1, 4).reshape(-1, 32, 3, 4, k // 32, 8).flatten(0, 1)[:m] for t in (want, got))
    return torch.equal(want.view(torch.int16), got.view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 33, 255, 257, 300])
@pytest.mark.parametrize("hidden", [512, 2048, 4096, 8192])
@pytest.mark.parametrize("fragments", [True, False])
def test_norms(m, hidden, fragments):
    assert K().add_rmsnorm_terms_possible(hidden)
    h, delta, w = randn(m, hidden, seed=m), randn(m, hidden, seed=m + 1), randn(hidden, seed=2)
    h[0, 3], delta[m - 1, 5] = 1e-38, 3e38
    want_h, want = h.clone(), torch.empty_like(h)
    K().add_rmsnorm(want_h, delta, w, want, 1e-6)
    rows = K().add_rmsnorm_terms(h, delta, w, 1e-6, fragments)
    assert torch.equal(h, want_h) and torch.equal(rows.x, want) and same(rows, fragments)
    K().add_rmsnorm(want_h, None, w, want, 1e-6)
    rows = K().add_rmsnorm_terms(h, None, w, 1e-6, fragments)
    assert torch.equal(rows.x, want) and same(rows, fragments)


@pytest.mark.gpu
def test_widths_without_a_form():
    assert not any(K().add_rmsnorm_terms_possible(n) for n in (96, 256, 2080, 1000, 16384))


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(130, 192, 64), (300, 704, 96), (33, 64, 32), (257, 6144, 256)])
@pytest.mark.parametrize("form", [5, 6, 7])
@pytest.mark.parametrize("fragments", [True, False])
def test_activations(monkeypatch, m, n, k, form, fragments):
    a, w = randn(m, k, seed=m), randn(n, k, seed=n)
    a[0, 0] = 3.0e38                                   # sums beyond what the split holds
    k_ = K()
    monkeypatch.setattr(k_, "f32_plan", lambda *_: form)
    rows = k_.gemm_f32(a, w, gate_pairs="silu", leave_terms=fragments)
    plain = k_.gemm_f32(a, w, gate_pairs="silu")
    assert torch.equal(rows.x.isnan(), plain.isnan()) and torch.equal(rows.x.nan_to_num(), plain.nan_to_num())
    # a row that is not finite has terms without a meaning: every other row's
    finite = plain.isfinite().all(1)
    assert finite[1:].all()
    keep = 0 if finite[0] else 1
    rows.x[:keep] = 0.0
    first = rows.terms.view(-1, n // 64, 3, 4, 32, 8)[0, :, :, :, 0] if fragments else rows.terms[0]
    if keep:
        first.zero_()
    assert same(rows, fragments)
    w2 = randn(160, n // 2, seed=5)
    assert torch.equal(k_.gemm_f32(rows, w2), k_.gemm_f32(rows.x, w2))


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [(16, 4, 128, 16), (8, 2, 64, 16), (12, 4, 32, 4)])
@pytest.mark.parametrize("fragments", [True, False])
def test_attention(monkeypatch, sizes, fragments):
    from jax_vllm_amd.parts import attention_backend

    from .test_f32_path import build_paged, run_step

    nq, nkv, d, page = sizes
    g = torch.Generator().manual_seed(d)
    lengths = [1500, 70, 1300]
    ks, vs = ([torch.randn(n, nkv, d, generator=g) for n in lengths] for _ in range(2))
    *pages, tables = build_paged(ks, vs, page)
    reqs = [(0, 1500), (1, 69), (0, 1300)]
    queries = [torch.randn(n, nq, d, generator=g) for _, n in reqs]
    plain = run_step(sizes, reqs, pages, tables, queries)
    left = []
    run = attention_backend.run
    monkeypatch.setattr(attention_backend, "run", lambda *a: left.append(run(*a, terms=fragments)))
    assert torch.equal(run_step(sizes, reqs, pages, tables, queries), plain)
    assert isinstance(left[0], K().TermRows) and torch.equal(left[0].x.cpu(), plain) and same(left[0], fragments)
