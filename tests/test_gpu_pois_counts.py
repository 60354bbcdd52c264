"""State::likelihood of counts around the end of the log-factorial table, in an
instance that holds no impossible event and so a sum of its terms' own size."""
import math

import numpy as np
import pytest

from beep_amd import _lib, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 62, 63, 64, 65, 5000])
def test_state_likelihood_of_large_counts(gpu_lib, count):
    spec, truth = configs.seir_areas(4, 4, 30, seed=4, daily_obs=True)
    ctx = _lib.Context(spec, capacity=2, nslot=1)
    ctx.set_param([0], truth[None, :])
    ctx.simulate([0, 1], [0, 0], [1, 2], seed=6)
    tn = ctx.get_transnum(1)
    lam = ctx.get_transmean(1)
    # The last step changes no later mean: its counts are set freely where means are positive.
    where = lam[-1] > 0
    assert where.sum() >= 8
    tn[-1][where] = count
    ctx.put_transnum(1, 0, tn)
    n, lam = ctx.get_transnum(1).reshape(-1), ctx.get_transmean(1).reshape(-1).astype(np.float64)
    assert (n == count).sum() >= 8 and np.all(n[lam == 0] == 0)
    terms = []
    for k, m in zip(n[lam > 0], lam[lam > 0]):
        terms += [k * math.log(m), -m, -math.lgamma(k + 1.0)]
    # Each part to some 4 x 2^-53 of itself, the sum of fewer than 2,000 terms to 12 roundings of partial sums
    # (64 lanes x 4 wavefronts, eight to a thread): 2^-49 of the parts' magnitudes.
    tol = 2.0 ** -49 * sum(abs(t) for t in terms)
    got = ctx.pois_loglik([1])[0]
    assert abs(got - math.fsum(terms)) <= tol, (got, math.fsum(terms), tol)
    ctx.close()
