"""Tiles of 32 and of 64 columns of the dense contraction: a product with few
rows (32 columns) against the same rows of a larger one (64 columns), bit for
bit, from the smallest product to the last below the change (432 tiles of
64 x 64)."""
import numpy as np
import pytest

from beep_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,rows", [(64, 1), (64, 64 * 431), (128, 33), (128, 64 * 215), (320, 65), (320, 64 * 86 - 5)])
def test_tile_widths_agree(gpu_lib, K, rows):
    rng = np.random.default_rng(K + rows)
    more = 64 * (512 // (K // 64) + 1)                 # at least 512 tiles of 64 x 64
    A = rng.standard_normal((max(rows, more), K)).astype(np.float32)
    B = rng.standard_normal((K, K)).astype(np.float32)
    assert np.array_equal(_lib.debug_gemm(A[:rows], B), _lib.debug_gemm(A, B)[:rows])
