"""A batch's streams: the first batch of a device's first context is no slower
than later ones by streams that it does not pay for, and batches give the same
on ordinary streams, on masked ones and while those are being made."""
import threading
import time

import numpy as np
import pytest

from beep_amd import _lib, configs

pytestmark = pytest.mark.gpu


def _contexts(days, n=12):
    out = []
    for i in range(n):
        spec, truth = configs.seir_areas((3, 10, 25, 60, 100, 200)[i % 6], (1, 4)[i // 6], days, seed=2)
        ctx = _lib.Context(spec, capacity=3, nslot=1)
        ctx.set_param([0], truth[None, :])
        ctx.simulate([2], [0], [5 + i], seed=3)
        out.append(ctx)
    return out


def _batch(ctxs):
    items = [(c, _lib.WORK_SIMULATE, 0, 0, 0, 5 + i, 0, c.S) for i, c in enumerate(ctxs)]
    t0 = time.perf_counter()
    _lib.run_batch(items, seed=3)
    return time.perf_counter() - t0


def test_first_batch_of_short_launches(gpu_lib):
    best = 1e9
    for _ in range(3):
        ctxs = _contexts(20)
        first = _batch(ctxs)
        best = min(best, first - min(_batch(ctxs) for _ in range(4)))
        for c in ctxs:
            c.close()
    assert best < 0.015, best                   # a dozen masked streams take 40 ms and more


def test_batches_give_the_same_as_streams_are_made(gpu_lib):
    ctxs = _contexts(400)
    want = [c.get_transnum(2) for c in ctxs]
    for _ in range(12):                         # some 3 ms each: masked streams are made on the way
        _batch(ctxs)
        for c, w in zip(ctxs, want):
            assert np.array_equal(c.get_transnum(0), w)
    for c in ctxs:
        c.close()


def test_threads_while_streams_are_made(gpu_lib):
    """Three threads' batches of four launches, some 3 ms each, from no streams
    to masked ones, with contexts made and closed beside them."""
    ctxs = _contexts(400)
    want = [c.get_transnum(2) for c in ctxs]
    small, truth = configs.seir_areas(3, 1, 10, seed=2)
    wrong = []

    def work(k):
        mine = ctxs[4 * k: 4 * k + 4]
        items = [(c, _lib.WORK_SIMULATE, 0, 0, 0, 5 + 4 * k + i, 0, c.S) for i, c in enumerate(mine)]
        for _ in range(15):
            _lib.run_batch(items, seed=3)
            extra = _lib.Context(small, capacity=1, nslot=1)
            for c, w in zip(mine, want[4 * k:]):
                if not np.array_equal(c.get_transnum(0), w):
                    wrong.append(k)
            extra.close()

    th = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in th:
        t.start()
    for t in th:
        t.join(timeout=90)
        assert not t.is_alive()
    assert not wrong
    for c in ctxs:
        c.close()
