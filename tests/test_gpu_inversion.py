"""Small-mean Poisson draws against the exact quantile of their uniform, over
enough draws (4 million per mean) that uniforms within a few 2^-24 of one
occur: there the FP32 sum can stop growing below the uniform."""
import numpy as np
import pytest

from beep_amd import _lib

pytestmark = pytest.mark.gpu


def _philox_word0(cells, key, seed):
    """First word of Philox-4x32-10 on counters (0, cell, 0x80000000, key)."""
    m0, m1, mask = np.uint64(0xD2511F53), np.uint64(0xCD9E8D57), np.uint64(0xFFFFFFFF)
    c = [np.zeros(len(cells), np.uint64), cells.astype(np.uint64), np.full(len(cells), 0x80000000, np.uint64),
         np.full(len(cells), key, np.uint64)]
    k0, k1 = seed & 0xFFFFFFFF, seed >> 32
    for _ in range(10):
        p0, p1 = m0 * c[0], m1 * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & mask, (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), p0 & mask]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return c[0]


@pytest.mark.parametrize("lam", [1e-8, 1e-3, 0.5, 4.0, 9.9999])
def test_inversion_quantiles(gpu_lib, lam):
    n, key, seed = 1 << 22, 77, 20250107
    lam32 = np.float32(lam)
    got = _lib.debug_poisson(np.full(n, lam32, np.float32), seed=seed, key=key)
    u = ((_philox_word0(np.arange(n), key, seed) >> np.uint64(8)).astype(np.float64) + 0.5) * 2.0 ** -24
    assert u.max() > 1 - 2.0 ** -20
    k = np.arange(1, 66)
    pmf = np.exp(-np.float64(lam32)) * np.concatenate([[1.0], np.cumprod(np.float64(lam32) / k)])
    cdf = np.cumsum(pmf)
    # FP32: at most 64 sums rounded to 2^-25 and terms of relative error below
    # 40 x 2^-24 in all: 64 x 3e-8 + 40 x 6e-8 < 4.4e-6.
    tol = 4.4e-6
    assert got.min() >= 0 and got.max() <= 64
    assert np.all(u <= np.minimum(cdf[got], 1.0) + tol)
    lower = np.where(got > 0, cdf[np.maximum(got - 1, 0)], -1.0)
    assert np.all(u > lower - tol)
