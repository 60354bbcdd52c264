"""Calls of a context whose HBM budget leaves no room for more scratch: what
has a way to do with less gives the results of a context without a budget,
keeps the scratch that was held and leaves no error text behind."""
import numpy as np
import pytest

from beep_amd import _lib, configs, spec as specmod

pytestmark = pytest.mark.gpu


def _error(ctx):
    return _lib.lib().beep_last_error(ctx._h).decode()


def _pair(spec, capacity, start, **kw):
    """Two contexts after start(ctx): one without a budget, one whose budget is
    what the first then holds."""
    free = _lib.Context(spec, capacity=capacity, nslot=1, **kw)
    start(free)
    tight = _lib.Context(spec, capacity=capacity, nslot=1, hbm_budget=free.device_bytes, **kw)
    start(tight)
    assert tight.device_bytes == free.device_bytes
    return free, tight


@pytest.mark.parametrize("keep", [_lib.KEEP_ALL, _lib.KEEP_TRANSNUM | _lib.KEEP_TRANSMEAN])
def test_transfers_within_held_scratch(gpu_lib, keep):
    """Trajectories of 60 steps move through the scratch that is there."""
    spec, truth = configs.seir_areas(100, 4, 60, seed=3, daily_obs=True)

    def start(ctx):
        ctx.set_param([0], truth[None, :])
        ctx.simulate([0], [0], [5], seed=4)
        ctx.obs_loglik([0])                         # takes the first 64 KB of scratch: 13 steps

    free, tight = _pair(spec, 2, start, keep=keep)
    held = tight.device_bytes
    for ctx in (free, tight):
        ctx.tn = ctx.get_transnum(0)
        ctx.put_transnum(1, 0, ctx.tn)
        ctx.tm = ctx.get_transmean(1)
    assert free.device_bytes > held                 # the slabs wanted more than was held
    assert tight.device_bytes == held
    assert _error(tight) == ""
    assert np.array_equal(free.tn, tight.tn)
    assert np.array_equal(free.tm.view(np.int32), tight.tm.view(np.int32))
    assert np.array_equal(free.get_state(1), tight.get_state(1))
    free.close()
    tight.close()


def test_copies_without_scratch(gpu_lib):
    """Lists of independent pairs need no memory."""
    spec, truth = configs.seir_areas(9, 4, 12, seed=3, daily_obs=True)

    def start(ctx):
        ctx.set_param([0], truth[None, :])
        ctx.simulate(range(6), [0] * 6, range(5, 11), seed=4)

    free, tight = _pair(spec, 6, start)
    held = tight.device_bytes
    for ctx in (free, tight):
        ctx.copy_instances([3, 4, 5], [0, 1, 0])
        ctx.copy_states([1, 2], [4, 0])
    assert free.device_bytes > held and tight.device_bytes == held
    assert _error(tight) == ""
    for i in range(6):
        for get in ("get_transnum", "get_transmean", "get_pop", "get_state"):
            assert np.array_equal(getattr(free, get)(i), getattr(tight, get)(i)), (get, i)
    free.close()
    tight.close()


@pytest.mark.parametrize("n", [512, 5461])
def test_state_likelihood_within_held_scratch(gpu_lib, n):
    """18 chunks of elements an instance: the chunk sums of 512 instances pass
    64 KB, 5,461 results alone fill it."""
    spec, truth = configs.seir_areas(100, 4, 60, seed=3, daily_obs=True)

    def start(ctx):
        ctx.set_param([0], truth[None, :])
        ctx.simulate(range(5), [0] * 5, range(5, 10), seed=4)
        ctx.obs_loglik([0])                         # takes the first 64 KB of scratch

    free, tight = _pair(spec, 5, start)
    held = tight.device_bytes
    ids = np.arange(n) % 5
    a, b = free.pois_loglik(ids), tight.pois_loglik(ids)
    assert free.device_bytes > held and tight.device_bytes == held
    assert _error(tight) == ""
    if n == 512:
        assert np.array_equal(a, b)                 # the same chunks, fewer instances at a time
    else:
        # One sum of 72,000 terms instead of 18: 72,000 x 2^-53 of the terms' magnitude (about |a|, all of one sign
        # but for log lam above 1).
        assert np.all(np.abs(a - b) <= 1e-10 * np.abs(a))
    free.close()
    tight.close()


@pytest.mark.parametrize("dt", [True, False])
def test_observations_within_held_scratch(gpu_lib, dt):
    """2,000 instances of two data tables: their chunk sums pass 64 KB, the sums
    of whole lists do not; the error functions are stored either way."""
    spec, truth = configs.seir_areas(12, 1, 30, seed=3, daily_obs=True)
    spec = specmod.expand_obs(spec)
    for k, o in enumerate(spec["obs"]):
        o["datatable"] = k % 2

    def start(ctx):
        ctx.set_param([0], truth[None, :])
        ctx.simulate(range(5), [0] * 5, range(5, 10), seed=4)
        ctx.obs_loglik([0])                         # takes the first 64 KB of scratch

    free, tight = _pair(spec, 5, start)
    held = tight.device_bytes
    ids = np.arange(2000 if dt else 4800) % 5
    a, b = free.obs_loglik(ids, with_dt=dt), tight.obs_loglik(ids, with_dt=dt)
    assert free.device_bytes > held and tight.device_bytes == held
    assert _error(tight) == ""
    if dt:
        assert np.all(np.abs(a[1] - b[1]) <= 1e-12 * np.abs(a[1]))      # a few hundred FP64 terms of one sign
        a, b = a[0], b[0]
    assert np.all(np.abs(a - b) <= 1e-12 * np.abs(a))
    pairs = [0, 1, 2, 3, 4], [1, 2, 3, 4, 0]
    acc = [ctx.accept(*pairs, mode=1, dlogq=np.zeros(5), key=np.arange(5), invT=1e-3)[0] for ctx in (free, tight)]
    # exp of invT / 2 times differences of error functions, each to 1e-12 of its size.
    assert np.all(np.abs(acc[0] - acc[1]) <= 1e-12 * (1 + 2 * np.abs(a).max()) * acc[0])
    assert len(set(np.round(acc[0], 12))) > 2
    free.close()
    tight.close()


def test_context_without_room_for_table_lists(gpu_lib):
    """The data tables' lists are 625 KB of a context that a budget without them
    still serves."""
    spec, truth = configs.seir_areas(400, 1, 400, seed=3, daily_obs=True)
    spec = specmod.expand_obs(spec)
    for k, o in enumerate(spec["obs"]):
        o["datatable"] = k % 2
    lists = 4 * len(spec["obs"])
    assert lists == 640000
    free = _lib.Context(spec, capacity=3, nslot=1)
    tight = _lib.Context(spec, capacity=3, nslot=1, hbm_budget=free.device_bytes - lists + 500000)
    assert tight.device_bytes == free.device_bytes - lists and _error(tight) == ""
    out = []
    for ctx in (free, tight):
        ctx.set_param([0], truth[None, :])
        ctx.simulate(range(3), [0] * 3, range(5, 8), seed=4)
        out.append(ctx.obs_loglik([2, 0, 1], with_dt=True))
    assert _error(tight) == ""
    for a, b in zip(*out):
        # 160,000 terms in another order: to 160,000 x 2^-53 of their magnitudes, at most some five times the sum.
        assert np.all(np.abs(a - b) <= 1e-10 * np.abs(a))
    assert np.array_equal(free.obs_loglik([1]), tight.obs_loglik([1]))
    free.close()
    tight.close()
