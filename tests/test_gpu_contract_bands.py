"""Tiles of 32 columns of the dense contraction up to 384 tiles of 64 x 64 and
above 512, of 64 columns between: products and simulations on both sides of
either edge give the same, bit for bit."""
import numpy as np
import pytest

from beep_amd import _lib, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,tiles", [(64, (384, 385, 512, 513)), (320, (380, 385, 510, 515)), (128, (2, 400, 1026))])
def test_products_across_the_bands(gpu_lib, K, tiles):
    rng = np.random.default_rng(K)
    rows = [64 * t // (K // 64) - 7 for t in tiles]
    A = rng.standard_normal((max(rows), K)).astype(np.float32)
    B = rng.standard_normal((K, K)).astype(np.float32)
    want = _lib.debug_gemm(A, B)
    for r in rows[:-1]:
        assert np.array_equal(_lib.debug_gemm(A[:r], B), want[:r]), r


def test_simulations_across_the_bands(gpu_lib):
    """20 areas in one column of tiles: 100 particles of nine groups are 15 tiles,
    2,800 are 394, 3,700 are 521."""
    spec, truth = configs.dense_pmcmc(A=20, period=6, with_obs=False)
    n = 3700
    ctx = _lib.Context(spec, capacity=n, nslot=1)
    ctx.set_param([0], truth[None, :])
    look = [0, 63, 99, 1500, 2799, 3699]
    got = []
    for m in (3700, 2800, 100):
        ids = np.arange(m)
        ctx.simulate(ids, ids * 0, ids + 1, seed=8)
        got.append({i: (ctx.get_transnum(i), ctx.get_transmean(i)) for i in look if i < m})
    assert sum(int(got[0][i][0].sum()) for i in look) > 0
    for g in got[1:]:
        for i, (tn, tm) in g.items():
            assert np.array_equal(tn, got[0][i][0]) and np.array_equal(tm, got[0][i][1]), i
    ctx.close()
