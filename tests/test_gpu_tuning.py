"""Tuned workgroup sizes of mixed batches: each specialised kernel of a size
class has its own, and a saved table is used only by the kernels that it was
tuned for."""
import os
import subprocess
import sys

import numpy as np
import pytest

from beep_amd import _lib, configs

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _launches(ctx, **kw):
    n = _lib.run_batch([(ctx, _lib.WORK_SIMULATE, i, 0, 0, 5 + i, 0, ctx.S) for i in range(2)], seed=3, stream=1, **kw)[1]
    return int(n)


def test_each_kernel_is_tuned(gpu_lib):
    """One structure and size, kernels compiled for other trajectories: the
    first tuned does not decide for the second."""
    spec, truth = configs.seir_areas(50, 9, 20, seed=2)
    out = []
    for keep in (_lib.KEEP_TRANSNUM | _lib.KEEP_POP, _lib.KEEP_TRANSNUM):      # tuned by no other test
        ctx = _lib.Context(spec, capacity=2, nslot=1, keep=keep)
        ctx.set_param([0], truth[None, :])
        plain = _launches(ctx)
        want = ctx.get_transnum(1)
        tuned, again = _launches(ctx, autotune=True), _launches(ctx, autotune=True)
        assert plain == again == 1
        assert tuned >= 3, keep                                   # 64, 128, 256 and 512 threads
        assert np.array_equal(ctx.get_transnum(1), want)
        out.append(want)
        ctx.close()
    assert np.array_equal(*out)


RUN = """
from beep_amd import _lib, configs
spec, truth = configs.seir_areas(30, 4, 10, seed=2)
ctx = _lib.Context(spec, capacity=1, nslot=1)
ctx.set_param([0], truth[None, :])
print(int(_lib.run_batch([(ctx, _lib.WORK_SIMULATE, 0, 0, 0, 5, 0, ctx.S)], autotune=True)[1]))
"""


def test_saved_sizes_of_other_kernels_are_ignored(gpu_lib, tmp_path):
    path = tmp_path / "tune.txt"

    def launches():
        env = dict(os.environ, BEEP_TUNE_CACHE=str(path))
        r = subprocess.run([sys.executable, "-c", RUN], cwd=ROOT, env=env, capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stderr
        return int(r.stdout.split()[-1])

    assert launches() == 2                          # 64 and 128 threads
    saved = path.read_text()
    assert launches() == 1                          # taken from the file
    head, _, rest = saved.partition("\n")
    for other in (head.split()[0] + " 0123456789abcdef", "beep-tune-3"):
        path.write_text(other + "\n" + rest)
        assert launches() == 2
        assert path.read_text().startswith(head + "\n")
