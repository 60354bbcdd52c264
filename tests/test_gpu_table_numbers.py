"""Data tables with few observations and high numbers: a context is made in the
time its observations take, and sums per table are those of the same
observations under low numbers."""
import time

import numpy as np
import pytest

from beep_amd import _lib, configs, spec as specmod

pytestmark = pytest.mark.gpu


def test_high_table_numbers(gpu_lib):
    spec, truth = configs.seir_areas(400, 1, 120, seed=3, daily_obs=True)
    spec = specmod.expand_obs(spec)
    n = len(spec["obs"])
    assert n == 48000
    low, high = [0, 1, 2], [7, 500000, 999999]
    out, took = [], []
    for numbers in (low, high):
        for k, o in enumerate(spec["obs"]):
            o["datatable"] = numbers[k % 3 if k < n - 1 else 2]
        _lib.Context(spec, capacity=1, nslot=1).close()       # compiles the kernels
        t0 = time.perf_counter()
        ctx = _lib.Context(spec, capacity=1, nslot=1)
        took.append(time.perf_counter() - t0)
        ctx.set_param([0], truth[None, :])
        ctx.simulate([0], [0], [5], seed=4)
        L, EF = ctx.obs_loglik([0], with_dt=True)
        out.append((L[0], EF[0]))
        ctx.close()
    assert took[1] < 2 * took[0] + 1.0, took
    (La, Ea), (Lb, Eb) = out
    assert La == Lb and Ea.shape == (3,) and Eb.shape == (1000000,)
    assert np.array_equal(Eb[high], Ea) and np.count_nonzero(Eb) == 3
