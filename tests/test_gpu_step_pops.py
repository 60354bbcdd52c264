"""Populations of the step-wise path's specialised transition kernel: between
steps they live in the kept trajectory, and without one in the state.  Both,
whole, in sections (sizes of one step among them) and step by step, against
the generic transition kernel."""
import numpy as np
import pytest

from beep_amd import _lib, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("keep", [_lib.KEEP_ALL, _lib.KEEP_TRANSNUM | _lib.KEEP_TRANSMEAN, _lib.KEEP_TRANSNUM | _lib.KEEP_POP])
@pytest.mark.parametrize("areas", [28, 29])     # 252 and 261 cells: one workgroup, and one more of five cells
def test_step_populations(gpu_lib, keep, areas):
    spec, truth = configs.dense_pmcmc(A=areas, period=40, with_obs=False)
    a = _lib.Context(spec, capacity=3, nslot=1, keep=keep | _lib.STEPWISE)
    b = _lib.Context(spec, capacity=3, nslot=1, keep=keep | _lib.STEPWISE | _lib.GENERIC_KERNEL)
    assert a.path == _lib.PATH_STEPWISE_SPEC and b.path == _lib.PATH_STEPWISE
    S = a.get_transnum(0).shape[0]
    for ctx in (a, b):
        ctx.set_param([0], truth[None, :])
        ctx.simulate([0], [0], [5], seed=3, stream=1)
        for t0, t1 in ((0, 1), (1, S // 2), (S // 2, S // 2), (S // 2, S - 1), (S - 1, S)):
            ctx.simulate([1], [0], [5], t0, t1, seed=3, stream=1)
        ctx.simulate([2], [0], [5], seed=3, stream=1, plain=True)
    for i in range(3):
        assert np.array_equal(a.get_transnum(i), a.get_transnum(0))
        assert np.array_equal(a.get_transnum(i), b.get_transnum(i))
        assert np.array_equal(a.get_state(i), b.get_state(i))
        if keep & _lib.KEEP_POP:
            assert np.array_equal(a.get_pop(i), b.get_pop(i))
        if keep & _lib.KEEP_TRANSMEAN:
            assert np.array_equal(a.get_transmean(i), b.get_transmean(i))
    a.close()
    b.close()
