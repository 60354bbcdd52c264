"""Coupled proposals with masks on the step-wise path's specialised transition
kernel, over one and several workgroups of cells, against the generic kernel
and, where mixing is sparse, the fused one."""
import numpy as np
import pytest

from beep_amd import _lib, configs, spec as specmod

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("keep", [_lib.KEEP_ALL, _lib.KEEP_TRANSNUM | _lib.KEEP_TRANSMEAN])
@pytest.mark.parametrize("dense,areas", [(True, 28), (True, 29), (True, 86), (False, 30), (False, 100)])
def test_masked_proposals(gpu_lib, keep, dense, areas):
    """252 cells and 261, 774, 270 and 900: one workgroup of 256, and more."""
    if dense:
        spec, truth = configs.dense_pmcmc(A=areas, period=40, with_obs=False)
    else:
        spec, truth = configs.seir_areas(areas, 9, 40, seed=3)
    n = 4
    keeps = [keep | _lib.STEPWISE, keep | _lib.STEPWISE | _lib.GENERIC_KERNEL] + ([] if dense else [keep])
    rng = np.random.default_rng(areas)
    params = np.concatenate([truth[None, :], specmod.sample_prior(spec, rng, 2 * n - 1)])
    inst = np.arange(n)
    ref = None
    for kp in keeps:
        ctx = _lib.Context(spec, capacity=2 * n, nslot=2 * n, keep=kp)
        if ref is None:
            mask = (rng.uniform(size=(n, ctx.S, ctx.A)) < 0.3).astype(np.uint8)
            mask[0], mask[1] = 0, 1                           # none and all simulated afresh
            mask[2, :, : ctx.A // 2] = 0
        ctx.set_param(range(2 * n), params)
        ctx.simulate(inst, inst, 40 + inst, seed=3, stream=6)
        ctx.mbp(inst, n + inst, n + inst, 90 + inst, simu_mask=mask, seed=4, stream=8)
        got = []
        for i in range(2 * n):
            got += [ctx.get_transnum(i), ctx.get_transmean(i), ctx.get_state(i)]
            if keep & _lib.KEEP_POP:
                got.append(ctx.get_pop(i))
        ctx.close()
        if ref is None:
            ref = got
            assert sum(int(g.sum()) for g in got[::len(got) // (2 * n)]) > 0
        else:
            for a, b in zip(ref, got):
                assert np.array_equal(a, b), kp
