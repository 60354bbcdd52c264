"""Section log-likelihoods summed in chunks of 2,048 observations, and the
bootstrap with its work arrays in LDS (up to 2,048 particles) and in memory."""
import numpy as np
import pytest

from beep_amd import _lib, configs
from oracle import oracle as O
from test_gpu_pmcmc import _device_uniforms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("days", [1, 16, 17, 40])        # 128 areas: 128, 2048, 2176 and 5120 observations
@pytest.mark.parametrize("n", [1, 5])
def test_section_chunks(gpu_lib, days, n):
    spec, truth = configs.seir_areas(128, 4, 60, seed=4, daily_obs=True)
    spec["sections"] = [(0, days), (days, 60)]
    ctx = _lib.Context(spec, capacity=n, nslot=1)
    ctx.set_param([0], truth[None, :])
    inst, key = np.arange(n), 3 + np.arange(n)
    ob, bp = ctx.pmcmc_obs_prob(inst[:1], 0, key[:1], invT=1.0, seed=9, stream=2)
    ctx.simulate(inst, np.zeros(n, int), key, seed=9, stream=2)
    L = [ctx.obs_loglik(inst, section=k) for k in range(2)]
    # One particle: the estimate is the sum of the sections' likelihoods.
    assert ob == L[0][0] + L[1][0]
    for k in range(2):
        whole, _ = ctx.obs_loglik(inst, section=k, with_dt=True)       # one chunk
        # Both add the same terms (all negative) in FP64, in another order.
        nobs = 128 * (days if k == 0 else 60 - days)
        assert np.all(whole < 0)
        assert np.all(np.abs(L[k] - whole) <= nobs * 2.0 ** -53 * np.abs(whole))
    ctx.close()


@pytest.mark.parametrize("n", [2047, 2048, 2049])
def test_bootstrap_work_arrays(gpu_lib, n):
    L = -50.0 + 3.0 * np.random.default_rng(n).standard_normal(n)
    bp, ob = _lib.bootstrap(L, 1.0, 5, 1, 2)
    bpo, obo = O.bootstrap(L, 1.0, _device_uniforms(n, 5, 1, 2))
    assert np.array_equal(bp, bpo)
    assert abs(ob - obo) <= 1e-12 * abs(obo)
