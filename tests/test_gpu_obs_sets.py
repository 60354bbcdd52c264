"""Log-likelihoods of a batch over several contexts: each item's value is its
context's own, bit for bit, for instance counts around the groups of four,
lists shorter and longer than a chunk, a context without observations and
contexts of different kernel variants in one call."""
import numpy as np
import pytest

from beep_amd import _lib, configs, spec as specmod

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [(1, 1, 1, 1), (4, 9, 3, 5), (8, 2, 7, 1)])
def test_batch_equals_contexts(gpu_lib, counts):
    models = [configs.seir_areas(3, 1, 40, seed=2, daily_obs=True),         # 120 observations
              configs.seir_areas(60, 4, 50, seed=3, daily_obs=True),        # 3,000
              configs.seir_areas(5, 4, 30, seed=4),                         # none
              configs.seir_areas(20, 4, 50, seed=5, obs_every=7)]           # Poisson
    ctxs, items = [], []
    for (spec, truth), n in zip(models, counts):
        spec = specmod.expand_obs(spec)
        ctx = _lib.Context(spec, capacity=10, nslot=1)
        ctx.set_param([0], truth[None, :])
        ctxs.append(ctx)
        # Instances out of order, interleaved between the contexts below.
        items += [(ctx, _lib.WORK_SIMULATE, 9 - k, 0, 0, 30 + k, 0, ctx.S) for k in range(n)]
    order = np.random.default_rng(1).permutation(len(items))
    items = [items[k] for k in order]
    _stats, L = _lib.run_batch(items, seed=3, stream=2, loglik=True)
    for (ctx, _k, inst, *_), Li in zip(items, L):
        assert ctx.obs_loglik([inst])[0] == Li
    for ctx in ctxs:
        ctx.close()
