"""Sums per data table against the observation values and densities in numpy:
tables smaller and larger than a chunk of observations, a table without any,
and instance counts around a group of four."""
import numpy as np
import pytest

from beep_amd import _lib, configs, spec as specmod

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 4, 5])
@pytest.mark.parametrize("A,days,ntab", [(1, 20, 1), (30, 80, 3), (45, 100, 11)])
def test_table_sums(gpu_lib, A, days, ntab, n):
    spec, truth = configs.seir_areas(A, 4, days, seed=2, daily_obs=True)
    spec = specmod.expand_obs(spec)
    rng = np.random.default_rng(A + ntab)
    # The last table is the largest; table 1 (of more than two) holds nothing.
    tab = np.where(rng.random(len(spec["obs"])) < 0.9, ntab - 1, rng.integers(0, ntab, len(spec["obs"])))
    if ntab > 2:
        tab[tab == 1] = 0
    for o, t in zip(spec["obs"], tab):
        o["datatable"] = int(t)
    ctx = _lib.Context(spec, capacity=6, nslot=1)
    ctx.set_param([0], truth[None, :])
    ids = np.arange(6)
    ctx.simulate(ids, ids * 0, ids + 3, seed=8)
    L, E = ctx.obs_loglik(ids[:n], with_dt=True)
    plain = ctx.obs_loglik(ids[:n])
    y, sd = np.array([o["y"] for o in spec["obs"]]), np.array([o["sd"] for o in spec["obs"]])
    for i in range(n):
        v = ctx.obs_values(i)
        lp = -0.5 * np.log(2 * np.pi * sd ** 2) - (y - v) ** 2 / (2 * sd ** 2)
        scale = np.abs(lp).sum()
        # 4500 FP64 terms: each sum within 4500 x 2^-53 of its magnitude.
        for d in range(ntab):
            assert abs(E[i, d] + 2 * lp[tab == d].sum()) <= 1e-12 * scale
        assert abs(L[i] - lp.sum()) <= 1e-12 * scale
        assert abs(L[i] - plain[i]) <= 1e-12 * scale
    ctx.close()
