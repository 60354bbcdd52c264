"""Binomial draws by inversion are pinned count by count: checksums of 16.8
million draws per (n, p), taken of the search that steps through the masses one
by one.  Rounding a mass once less (a subtraction fused with the product before
it) moves a few draws at the edges between two counts and changes five of them."""
import zlib

import numpy as np
import pytest

from beep_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,p,crc", [(2, 0.5, 0x774dd415), (19, 0.5, 0xe0fbe24a), (19, 0.4999, 0x191bceb5),
                                     (40, 0.2, 0x7af24788), (37, 0.9, 0xc456a850), (300, 0.033, 0x30c0c49b),
                                     (12, 0.3, 0xbc019ce8), (90, 0.11, 0xc095b39c), (5000, 0.0019, 0x67ffd3f5)])
def test_binomial_counts(gpu_lib, n, p, crc):
    m = 1 << 24
    got = _lib.debug_binomial(np.full(m, n), np.full(m, float(np.float32(p))), seed=20250109, key=80)
    assert zlib.crc32(np.ascontiguousarray(got, dtype=np.int32).tobytes()) == crc
