"""State::likelihood against numpy on the device's own counts and means:
trajectories below, at and above a chunk of elements, counts above the
log-factorial table, and zero means with and without events."""
import math

import numpy as np
import pytest

from beep_amd import _lib, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("A,G,days", [(1, 1, 5), (1, 1, 300), (16, 4, 64), (33, 9, 40)])
def test_state_likelihood(gpu_lib, A, G, days):
    spec, truth = configs.seir_areas(A, G, days, seed=4, daily_obs=True)
    ctx = _lib.Context(spec, capacity=3, nslot=1)
    ctx.set_param([0], truth[None, :])
    ids = np.arange(3)
    ctx.simulate(ids, ids * 0, ids + 1, seed=6)
    tn = ctx.get_transnum(1)
    tn[0, 0, 2, 0] += 3                    # recoveries where the mean is zero at the first step
    tn[days // 2, 0, 0, 0] += 200          # a count above the table
    ctx.put_transnum(1, 0, tn)
    got = ctx.pois_loglik([2, 1, 0])
    for i, g in zip([2, 1, 0], got):
        n, lam = ctx.get_transnum(i).reshape(-1), ctx.get_transmean(i).reshape(-1).astype(np.float64)
        lg = np.array([math.lgamma(k + 1.0) for k in range(int(n.max()) + 1)])
        with np.errstate(divide="ignore", invalid="ignore"):
            lp = np.where(lam == 0, np.where(n == 0, 0.0, -1e9), np.where(n == 0, -lam, n * np.log(lam) - lam - lg[n]))
        # Terms to a few 1e-15 of their parts, sums of 12,000 terms to 12,000 x 2^-53.
        assert abs(g - math.fsum(lp)) <= 4e-12 * np.abs(lp).sum() + 1e-9 * (np.abs(lp) < 1e8).sum() * 1e-6
    ctx.close()
