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


def test_where_a_wave_walks_several_tiles():
    from jax_vllm_amd.ops.kernels import head_walk

    # a tile a wave: steps filled up with zeros, one step, an inner size that registers do not hold
    assert [head_walk(4096, 64, K, 64, False) for K in (16, 32, 56, 72, 96, 160, 216, 264, 512)] == [0] * 9
    assert all(head_walk(4096, 64, K, 64, False) == 4 for K in (64, 128, 192, 224, 232, 256))
    # one block a unit, rounded down; twice as many with gates, unless these have less than one and a half tiles a wave
    assert head_walk(600, 192, 256, 16, False) == 5 and head_walk(600, 192, 256, 16, True) == 5 and head_walk(1024, 192, 256, 16, True) == 10
    assert head_walk(1216, 192, 256, 16, True, cus=304) == 12 and head_walk(2048, 64, 224, 16, True) == 16
    assert [head_walk(n, 64, 128, 16, False) for n in (1472, 1473, 1536, 1537)] == [0, 16, 16, 16]
    assert head_walk(80, 64, 64, 64, False) == 2 and head_walk(80, 64, 128, 64, False) == 0
    assert head_walk(64 * 200, 40, 64, 400, True) == 1 and head_walk(0, 64, 64, 1, False) == 0 and head_walk(5, 64, 64, 0, False) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("n,heads,N,K", [(1100, 30, 72, 192), (1100, 30, 72, 232), (1600, 40, 40, 64), (2100, 16, 64, 224)])
@pytest.mark.parametrize("gate", [None, "element", "head"])
def test_walks_by_the_rule(n, heads, N, K, gate):
    from jax_vllm_amd.ops.kernels import head_walk

    assert 0 < head_walk(n, N, K, heads, gate is not None) < -(-n // 64)
    test_several_tiles_a_wave(n, heads, N, K, gate)
