"""The order in which a norm adds the squares of four neighbours: a row's bits hang on it, and steps whose kernels stand for one another have to agree."""
import numpy as np
import pytest
import torch

from .test_kernels_gpu import K


def _pairs(count):
    """(a, b, c): the float nearest to a^2 + float(b^2) is the float nearest to c^2, and float(a^2) + b^2 would round to another one."""
    rng, found = np.random.default_rng(1), []
    while len(found) < count:
        a, b = np.float32(rng.uniform(1, 2)), np.float32(rng.uniform(1, 2))
        # products of two floats are exact in 64 bits, and so are their sums with a float of this size
        here = np.float32(np.float64(a) * np.float64(a) + np.float64(b * b))
        there = np.float32(np.float64(a * a) + np.float64(b) * np.float64(b))
        c = np.float32(np.sqrt(np.float64(here)))
        if here != there and c * c == here:
            found.append((a, b, c))
    return found


@pytest.mark.gpu
@pytest.mark.parametrize("hidden", [256, 1024, 2048, 5120])
def test_the_second_square_of_a_piece_is_rounded_first(hidden):
    pairs, tiny = _pairs(64), 2.0 ** -40      # tiny: its square changes no sum, and times the scale it shows the scale's bits
    pieces, singles = (torch.zeros(64, hidden) for _ in range(2))
    for i, (a, b, c) in enumerate(pairs):
        pieces[i, 4], pieces[i, 5], singles[i, 6] = float(a), float(b), float(c)
    pieces[:, 60] = singles[:, 60] = tiny
    weight, scales = torch.ones(hidden, device="cuda"), []
    for h in (pieces, singles):
        out = torch.empty(64, hidden, device="cuda")
        K().add_rmsnorm(h.cuda(), None, weight, out, 1e-6)
        scales.append(out[:, 60])
    assert torch.equal(*scales)
