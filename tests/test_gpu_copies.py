"""Instance and state copies: lists whose pairs are independent (one launch),
lists where a row is read and written or written twice (in order), pairs of an
instance with itself, and rows of odd length, against the same copies done in
order on the host."""
import numpy as np
import pytest

from beep_amd import _lib, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("A,G", [(1, 1), (3, 1), (4, 4), (37, 9)])
@pytest.mark.parametrize("dst,src", [([4, 5, 6], [0, 1, 0]), ([7], [3]), ([3, 3], [0, 1]), ([1, 2, 3], [0, 1, 2]),
                                     ([0, 1], [1, 0]), ([2, 5, 2], [2, 1, 0]), ([], [])])
def test_copies_in_order(gpu_lib, A, G, dst, src):
    spec, truth = configs.seir_areas(A, G, 7, seed=3, daily_obs=True)
    n = 8
    ctx = _lib.Context(spec, capacity=n, nslot=1)
    ctx.set_param([0], truth[None, :])
    ids = np.arange(n)
    ctx.simulate(ids, ids * 0, ids + 5, seed=4)
    ctx.obs_loglik(ids)

    def read():
        return [(ctx.get_state(i), ctx.get_transnum(i), ctx.get_transmean(i), ctx.get_pop(i)) for i in range(n)]

    want = read()
    for d, s in zip(dst, src):
        want[d] = want[s]
    ctx.copy_instances(dst, src)
    got = read()
    for w, g in zip(want, got):
        for a, b in zip(w, g):
            assert np.array_equal(a, b)
    # States alone: the trajectories stay.
    ctx.simulate(ids, ids * 0, ids + 50, 0, 5, seed=4)
    want = read()
    states = [w[0] for w in want]
    for d, s in zip(dst, src):
        states[d] = states[s]
    ctx.copy_states(dst, src)
    got = read()
    for i in range(n):
        assert np.array_equal(got[i][0], states[i])
        assert np.array_equal(got[i][1], want[i][1])
    ctx.close()
