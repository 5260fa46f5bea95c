"""The per-head product of many rows whose waves walk several tiles with their rows of W in registers: inner sizes at the edges of the
forms, last tiles that only some waves have, last rows that do not fill one, against float64 and bit for bit against few rows."""
import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("n,heads,N,K", [(1003, 40, 40, 64), (1003, 40, 40, 8), (1100, 33, 72, 72), (1025, 64, 64, 128), (700, 30, 72, 224),
                                         (1041, 20, 200, 256), (705, 30, 72, 136), (700, 30, 72, 264)])
@pytest.mark.parametrize("gate", [None, "element", "head"])
def test_several_tiles_a_wave(n, heads, N, K, gate):
    from jax_vllm_amd.ops import kernels as K_

    side = -(-N // 64) * heads
    assert n * N * heads >= 480000 and (K > 256 or -(-n // 64) > -(-256 // side))      # more tiles than waves along the rows
    g = torch.Generator().manual_seed(n + K)
    x = torch.randn(n, heads * K, generator=g).bfloat16().cuda()
    w = (torch.randn(heads, N, K, generator=g) * K ** -0.5).bfloat16().cuda()
    gates = torch.randn(n, heads * N if gate == "element" else heads, generator=g).bfloat16().cuda() if gate else None

    def run(a, b):
        y = torch.zeros(b - a, heads * N, dtype=torch.bfloat16, device="cuda")
        K_.head_linear(y, N, x[a:b], K, w, gate=gates[a:b] if gate else None)
        return y

    y = run(0, n)
    want = torch.matmul(x.cpu().double().view(n, heads, K).transpose(0, 1), w.cpu().double().transpose(1, 2)).transpose(0, 1)
    if gate:
        want = want * torch.sigmoid(gates.cpu().double().view(n, heads, -1))
    # 8 bits of fraction for the result; float sums of K terms of size x w
    bound = 2.0 ** -8 * want.abs() + K * 2.0 ** -23 * x.abs().max().item() * w.abs().max().item()
    assert bool(((y.cpu().double().view(n, heads, N) - want).abs() <= bound).all())
    for a in range(0, n, 79):                                      # up to 79 rows: the form of a tile a wave
        assert torch.equal(run(a, min(a + 79, n)), y[a:a + 79])
