"""The gradient kernel at the edges of its work split (16 samples per matrix
tile, four wavefronts per block, at most 256 blocks) against the FP64 oracle
with the same forward roundings."""
import numpy as np
import pytest

from oracle import mlp_oracle as mo
from test_mlp_gpu import random_params

pytestmark = pytest.mark.gpu

dyn = pytest.importorskip("dynfd3dcuda_amd")
from dynfd3dcuda_amd import mlp  # noqa: E402


@pytest.mark.parametrize("n", [1, 15, 16, 17, 64, 65, 1040, 16384, 16385, 33000])
def test_gradient_sizes(n):
    """FP32 sums of n terms are off by less than 1e-5 of the gradient's norm.
    A first-layer value whose FP32 sum falls on the other side of a bfloat16
    rounding boundary (one in about 2^14 values) moves by 2^-8 of itself, one
    of the sample's 64: up to 2^-8 / 8 of that sample's gradient, which
    averages out over many samples.  Bound: 1e-4 of the norm, 1e-3 for fewer
    than 64 samples."""
    Fa, Ta = mo.synthetic_samples(33000, seed=21)
    P = random_params(Fa, Ta, 7)  # standardisation from the whole set
    F, T = Fa[:n], Ta[:n]
    loss, g = mlp.grad(P, F, T)
    lref, gref = mo.loss_grad(P, F, T, bf16=True)
    tol = 1e-4 if n >= 64 else 1e-3
    assert abs(loss - lref) <= tol * lref, (loss, lref)
    assert np.all(g[:10] == 0)
    for k in ("W1", "b1", "W2", "b2", "w3", "b3"):
        a, b = np.atleast_1d(mo.unpack(g)[k]), np.atleast_1d(mo.unpack(gref)[k])
        assert np.linalg.norm(a - b) <= tol * max(np.linalg.norm(b), 1e-3 * np.linalg.norm(gref)), k
