"""The ABC-SMC weight kernel at the edges of its split: odd and even numbers of
variables, previous generations around the split's size, a matrix that is not
symmetric (the quadratic form's upper triangle with the mirrored entries added
is the same form), and zero weights."""
import numpy as np
import pytest

from beep_amd import _lib
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_prev,n_new,nvar", [(15, 1, 1), (16, 256, 2), (17, 257, 3), (33, 40, 9), (600, 300, 21),
                                               (1001, 13, 31), (130, 30, 32)])
def test_weights_at_split_edges(gpu_lib, n_prev, n_new, nvar):
    rng = np.random.default_rng(n_prev * 100 + nvar)
    prev = 3.0 + rng.normal(0, 1, (n_prev, nvar))
    w = rng.uniform(0.2, 3.0, n_prev) * (rng.random(n_prev) > 0.2)
    w[0] = 1.0
    theta = prev[rng.integers(0, n_prev, n_new)] + rng.normal(0, 0.3, (n_new, nvar))
    Q = rng.normal(0, 1, (nvar, nvar))
    skew = rng.normal(0, 0.5, (nvar, nvar))
    M = Q @ Q.T / nvar + np.eye(nvar) + (skew - skew.T)
    logprior = rng.normal(-3, 1, n_new)
    got = _lib.abcsmc_weights(prev, w, theta, M, 0.7, logprior)
    # Each exponent is a sum of at most 32^2 products, below ~1e3 in magnitude
    # where it matters: 1e3 x 34 x 2^-53 < 4e-12 relative in a term.
    for i in range(0, n_new, max(1, n_new // 16)):
        want = O.abcsmc_weight(theta[i], prev, w, M, 0.7, logprior[i])
        assert abs(got[i] / want - 1) < 1e-11
