"""Mixed batches of more size classes than the device has batch streams, and
batches of two host threads at once: every result equals the single-context
call's with the same keys."""
import threading

import numpy as np
import pytest

from beep_amd import _lib, configs

pytestmark = pytest.mark.gpu

AREAS = [1, 2, 9, 17, 33, 65, 129]


def _contexts():
    out = []
    for A in AREAS:
        for G in (1, 4):
            spec, truth = configs.seir_areas(A, G, 25, seed=A * 10 + G, daily_obs=True)
            ctx = _lib.Context(spec, capacity=4, nslot=4)
            ctx.set_param(np.arange(4), np.array([truth, truth, truth * [1.1, 1, 1, 1], truth]))
            out.append(ctx)
    return out


def _reference(ctxs, key0):
    """Trajectories of the single-context calls: a simulation into instance 0,
    a proposal coupled to it into instance 1."""
    out = []
    for i, c in enumerate(ctxs):
        c.simulate([0], [0], [key0 + i], seed=9, stream=2)
        c.mbp([0], [1], [2], [key0 + 500 + i], seed=9, stream=3)
        out.append((c.get_transnum(0), c.get_transnum(1)))
    return out


def _batches(ctxs, key0, rounds=3):
    out = []
    for _ in range(rounds):
        _lib.run_batch([(c, _lib.WORK_SIMULATE, 2, 0, 0, key0 + i, 0, c.S) for i, c in enumerate(ctxs)], seed=9, stream=2)
        _lib.run_batch([(c, _lib.WORK_MBP, 3, 2, 2, key0 + 500 + i, 0, c.S) for i, c in enumerate(ctxs)] +
                       [(c, _lib.WORK_SIMULATE, 0, 0, 1, key0 + 900 + i, 0, c.S) for i, c in enumerate(ctxs)],
                       seed=9, stream=3)
        out.append([(c.get_transnum(2), c.get_transnum(3)) for c in ctxs])
    return out


def _same(want, got):
    for w, g in zip(want, got):
        for a, b in zip(w, g):
            assert np.array_equal(a, b)


def test_more_classes_than_streams(gpu_lib):
    ctxs = _contexts()
    want = _reference(ctxs, 100)
    for got in _batches(ctxs, 100):
        _same(want, got)
    for c in ctxs:
        c.close()


def test_two_threads(gpu_lib):
    sets = [_contexts(), _contexts()]
    want = [_reference(s, 1000 * (k + 1)) for k, s in enumerate(sets)]
    got = [None, None]

    def work(k):
        got[k] = _batches(sets[k], 1000 * (k + 1))

    th = [threading.Thread(target=work, args=(k,)) for k in (0, 1)]
    for t in th:
        t.start()
    for t in th:
        t.join(timeout=60)
    for k in (0, 1):
        assert got[k] is not None
        for g in got[k]:
            _same(want[k], g)
    for s in sets:
        for c in s:
            c.close()
