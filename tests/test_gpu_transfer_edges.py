"""Trajectories read back and loaded at the edge between the host's and the
device's reordering (8,192 runs of an area's groups, 65,536 values): the same
counts whichever way they went, against sums that the device makes itself."""
import numpy as np
import pytest

from beep_amd import _lib, configs

pytestmark = pytest.mark.gpu


# Counts of three transitions: 8,190, 8,196 and 8,190 runs, of nine groups 65,529 values (7,281 runs), 65,637 and
# 65,610; populations of four compartments: 8,148 and 8,240 runs.
@pytest.mark.parametrize("A,G,S", [(26, 1, 105), (4, 1, 683), (21, 4, 130), (3, 9, 809), (17, 9, 143), (27, 9, 90),
                                   (21, 4, 97), (20, 4, 103)])
def test_transfers_both_ways(gpu_lib, A, G, S):
    spec, truth = configs.seir_areas(A, G, S, seed=3)
    ctx = _lib.Context(spec, capacity=3, nslot=1)
    ctx.set_param([0], truth[None, :])
    ctx.simulate([0], [0], [7], seed=2)
    tn, tm, pop = ctx.get_transnum(0), ctx.get_transmean(0), ctx.get_pop(0)
    for tr in range(ctx.T):
        assert np.array_equal(ctx.sum_transnum([0], tr, 0, ctx.S)[0], tn[:, :, tr].sum(axis=(1, 2)))
    # Populations are what the counts make of them, areas and groups in their places.
    for s in range(ctx.S - 1):
        for c in range(ctx.C):
            into = sum(tn[s, :, t] for t in range(ctx.T) if spec["trans"][t]["to"] == c)
            out = sum(tn[s, :, t] for t in range(ctx.T) if spec["trans"][t]["from"] == c)
            assert np.array_equal(pop[s + 1, :, c], pop[s, :, c] + into - out)
    ctx.put_transnum(1, 0, tn)
    assert np.array_equal(ctx.get_transnum(1), tn)
    assert np.array_equal(ctx.get_transmean(1), tm)
    assert np.array_equal(ctx.get_pop(1), pop)
    ctx.close()
