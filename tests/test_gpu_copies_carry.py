"""What a copied instance carries with its trajectory: the error function that
acceptance reads, in lists of independent pairs and in ordered ones."""
import numpy as np
import pytest

from beep_amd import _lib, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("A", [3, 4])
@pytest.mark.parametrize("dst,src", [([4, 5, 6], [0, 1, 0]), ([7], [3]), ([3, 3], [0, 1]), ([1, 2, 3], [0, 1, 2]),
                                     ([0, 1], [1, 0])])
def test_error_functions_go_with_copies(gpu_lib, A, dst, src):
    """Instances of unlike parameters; al of a proposal from each to instance 8
    and back names its error function."""
    spec, truth = configs.seir_areas(A, 4, 20, seed=3, daily_obs=True)
    n = 9
    ctx = _lib.Context(spec, capacity=n, nslot=n)
    ctx.set_param(range(n), truth[None, :] * (1 + 0.01 * np.arange(n))[:, None])
    ctx.simulate(range(n), range(n), range(5, 5 + n), seed=4)
    L = ctx.obs_loglik(range(n))
    assert len(set(L)) == n
    T = 0.1 / np.abs(L - L[8]).max()

    def al():
        one = [ctx.accept([i], [8], 1, np.zeros(1), [1], invT=T)[0][0] for i in range(8)]
        two = [ctx.accept([8], [i], 1, np.zeros(1), [1], invT=T)[0][0] for i in range(8)]
        return list(zip(one, two))

    want = al()
    assert len(set(want)) == 8
    ctx.copy_instances(dst, src)
    for d, s in zip(dst, src):
        want[d] = want[s]
    assert al() == want
    ctx.close()
