"""Binomial draws by inversion (n * min(p, 1 - p) < 10) against the exact
quantile of their uniform, a million draws per (n, p): p at and beyond one
half, one trial, means at both ends, trial counts in the millions; lanes of
one wavefront with unlike (n, p)."""
import numpy as np
import pytest
from scipy import stats

from beep_amd import _lib
from test_gpu_inversion import _philox_word0

pytestmark = pytest.mark.gpu

PAIRS = [(1, 0.3), (1, 0.999), (2, 0.5), (19, 0.5), (19, 0.4999), (40, 0.2), (37, 0.9), (300, 0.033), (5000, 1e-6),
         (2000000, 4.9e-6)]
# FP32: at most 64 differences rounded to 2^-25 (1.9e-6), the first mass's
# exponent (up to 14, relative 3 x 2^-24 in log1pf, product and exponential:
# 2.5e-6), and ratios a / k - s, each within 3 x 2^-24 / (1 - k / (n + 1)), of
# which the mass-weighted sum over k stays below 10 x 2 x 1.8e-7 = 3.6e-6;
# p / q adds 10 x 1.5e-7.
TOL = 1.2e-5


def _check(got, n, p, u):
    flip = p > 0.5
    pp = np.where(flip, 1 - p, p)
    k = np.where(flip, n - got, got)
    assert k.min() >= 0 and np.all(k <= n)
    sure = u < 1 - TOL                      # above, the mass may run out and the draw be made again
    assert np.all((u <= stats.binom.cdf(k, n, pp) + TOL)[sure])
    assert np.all((u > stats.binom.cdf(k - 1, n, pp) - TOL)[sure])


@pytest.mark.parametrize("n,p", PAIRS)
def test_binomial_quantiles(gpu_lib, n, p):
    m, key, seed = 1 << 20, 78, 20250108
    p = float(np.float32(p))
    got = _lib.debug_binomial(np.full(m, n), np.full(m, p), seed=seed, key=key)
    u = ((_philox_word0(np.arange(m), key, seed) >> np.uint64(8)).astype(np.float64) + 0.5) * 2.0 ** -24
    _check(got, np.full(m, n), np.full(m, p), u)


def test_binomial_mixed_lanes(gpu_lib):
    m, key, seed = 1 << 18, 79, 5
    rng = np.random.default_rng(1)
    which = rng.integers(len(PAIRS), size=m)
    n = np.array([a for a, _ in PAIRS])[which]
    p = np.array([float(np.float32(b)) for _, b in PAIRS])[which]
    got = _lib.debug_binomial(n, p, seed=seed, key=key)
    u = ((_philox_word0(np.arange(m), key, seed) >> np.uint64(8)).astype(np.float64) + 0.5) * 2.0 ** -24
    _check(got, n, p, u)
