"""The library's own work stays off the null stream, which waits for the batch
streams: contexts are made and weights computed while another thread's batch
runs."""
import threading
import time

import numpy as np
import pytest

from beep_amd import _lib, configs

pytestmark = pytest.mark.gpu


def test_context_made_beside_a_batch(gpu_lib):
    """The batch is one long instance (some 25 ms); a context of a structure
    compiled before takes a few milliseconds."""
    spec, truth = configs.seir_areas(400, 9, 2000, seed=4, daily_obs=False)
    small, struth = configs.seir_areas(3, 4, 10, seed=1, daily_obs=True)
    big = _lib.Context(spec, capacity=1, nslot=1)
    big.set_param([0], truth[None, :])
    items = [(big, _lib.WORK_SIMULATE, 0, 0, 0, 5, 0, big.S)]
    _lib.Context(small, capacity=2, nslot=1).close()       # compiles the kernels
    _lib.run_batch(items, seed=9, stream=2)                # makes the stream
    t0 = time.perf_counter()
    _lib.run_batch(items, seed=9, stream=2)
    alone = time.perf_counter() - t0
    best = 1e9
    for _ in range(3):
        done = [0.0]

        def work():
            _lib.run_batch(items, seed=9, stream=2)
            done[0] = time.perf_counter()

        th = threading.Thread(target=work)
        t0 = time.perf_counter()
        th.start()
        time.sleep(0.1 * alone)
        ctx = _lib.Context(small, capacity=2, nslot=1)
        ctx.set_param([0], struth[None, :])
        ctx.simulate([0], [0], [5], seed=1)
        made = time.perf_counter()
        th.join(timeout=60)
        ctx.close()
        best = min(best, (made - t0) / (done[0] - t0))
    big.close()
    assert best < 0.6, best                                # 1 where it waits for the batch


def test_calls_beside_batches_give_the_same(gpu_lib):
    spec, truth = configs.seir_areas(60, 4, 80, seed=4, daily_obs=True)
    rng = np.random.default_rng(3)
    prev, theta = rng.standard_normal((300, 7)), rng.standard_normal((200, 7))
    w, lp, M = rng.random(300), rng.standard_normal(200), np.eye(7)
    L = rng.standard_normal(1500)

    def calls():
        ctx = _lib.Context(spec, capacity=2, nslot=1)
        ctx.set_param([0], truth[None, :])
        ctx.simulate([0, 1], [0, 0], [5, 6], seed=1)
        out = [ctx.get_transnum(0), ctx.get_state(1), ctx.obs_loglik([0, 1])]
        ctx.close()
        out.append(_lib.abcsmc_weights(prev, w, theta, M, 1.5, lp))
        out.extend(_lib.bootstrap(L, 0.7, seed=3, stream=1, sec=2))
        out.append(_lib.debug_binomial(np.full(500, 30), np.full(500, 0.2), seed=3, key=4))
        return out

    want = calls()
    base = _lib.Context(spec, capacity=8, nslot=1)
    base.set_param([0], truth[None, :])
    stop = threading.Event()

    def batches():
        while not stop.is_set():
            _lib.run_batch([(base, _lib.WORK_SIMULATE, k, 0, 0, k, 0, base.S) for k in range(8)], seed=9, stream=2)

    th = threading.Thread(target=batches)
    th.start()
    got = [calls() for _ in range(5)]
    stop.set()
    th.join(timeout=60)
    assert not th.is_alive()
    base.close()
    for g in got:
        for a, b in zip(want, g):
            assert np.array_equal(a, b)
