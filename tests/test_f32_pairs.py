"""The 32-bit product of up to 8 rows by pairs of steps: the bits of the other forms at the edges of its blocks, rounds and the inner size."""
import pytest
import torch

from .test_f32_split import bound, product
from .test_kernels_gpu import randn


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(1, 1, 4), (8, 8, 32), (7, 9, 36), (8, 2049, 64), (5, 2048, 1020), (3, 25, 2052), (8, 50, 2080), (2, 2056, 4128), (8, 23, 8228),
                                   (6, 2100, 1092)])
def test_pairs_of_steps(m, n, k):
    """Form 2 takes 8 rows of w up to 2,048 of them and 16 beyond, form 4 takes 24; form 3 has tiles of 32 x 16.  Steps beyond a round's
    64, 32 and 16 a half, an odd number of steps, a last one of 4 columns."""
    a, w = randn(m, k, seed=m), randn(n, k, seed=n + k)
    want = product(3, a, w)
    assert ((want.double() - a.double() @ w.double().T).abs() <= bound(a, w)).all()
    for form in (2, 4):
        assert torch.equal(product(form, a, w), want), form
