"""Replaying a simulated trajectory's counts gives the simulation's own
populations, means and state bit for bit, whatever else the model has (age
matrices that vary, groups, covariates, several steps a day) and whichever
trajectories the context keeps."""
import numpy as np
import pytest

import toml_models
from beep_amd import _lib, configs

pytestmark = pytest.mark.gpu


def _check(spec, pv, keep=_lib.KEEP_ALL):
    ctx = _lib.Context(spec, capacity=2, nslot=1, keep=keep)
    ctx.set_param([0], np.asarray(pv)[None, :])
    ctx.simulate([0], [0], [77], seed=5, stream=2)
    ctx.put_transnum(1, 0, ctx.get_transnum(0))
    assert np.array_equal(ctx.get_state(0), ctx.get_state(1))
    assert np.array_equal(ctx.get_transnum(0), ctx.get_transnum(1))
    if keep & _lib.KEEP_TRANSMEAN:
        a, b = ctx.get_transmean(0), ctx.get_transmean(1)
        assert np.array_equal(a.view(np.int32), b.view(np.int32))
    if keep & _lib.KEEP_POP:
        assert np.array_equal(ctx.get_pop(0), ctx.get_pop(1))
    ctx.close()


@pytest.mark.parametrize("A,G,days", [(1, 1, 1), (1, 1, 17), (63, 1, 33), (65, 4, 16), (171, 9, 40)])
@pytest.mark.parametrize("keep", [_lib.KEEP_ALL, _lib.KEEP_TRANSNUM, _lib.KEEP_TRANSNUM | _lib.KEEP_TRANSMEAN])
def test_replay_areas(gpu_lib, A, G, days, keep):
    spec, truth = configs.seir_areas(A, G, days, seed=A, daily_obs=False)
    _check(spec, truth, keep)


def test_replay_spatial_generic(gpu_lib):
    spec, truth = configs.spatial_abcsmc(A=40, period=50, with_obs=False)
    _check(spec, truth)
    _check(spec, truth, _lib.KEEP_ALL | _lib.GENERIC_KERNEL)


@pytest.mark.parametrize("mk", [toml_models.toml_seir_erlang, toml_models.toml_seird_branch, toml_models.toml_sir_3areas,
                                toml_models.toml_sird_ages, toml_models.toml_seir_sex_ages, toml_models.toml_sird_strains])
def test_replay_models(gpu_lib, mk):
    _check(*mk())


@pytest.mark.parametrize("groups", [False, True])
def test_replay_groups_and_modifications(gpu_lib, groups):
    spec, truth = configs.seir_areas(12, 4, 30, seed=6, daily_obs=False)
    if groups:
        spec["R_splines"] = [{"spline": 0, "areas": list(range(5))}, {"spline": 0, "areas": list(range(5, 12))}]
    else:
        spec["modifications"] = [{"type": "trans_rate_fac", "start": 5, "end": 20, "factor": 1.7, "trans": [1], "areas": [2, 3]},
                                 {"type": "beta_fac", "start": 3, "end": 25, "factor": 0.6, "areas": [1, 2], "dps": [0]}]
    _check(spec, truth)
