"""Reads on both sides of the size from which a read goes through the pinned
ring: below it, one slot short of and past the ring, and a partial last slot."""

import numpy as np
import pytest

import kernrt_amd as K

pytestmark = pytest.mark.gpu

SLOT, LARGE = (2 << 20) // 4, (4 << 20) // 4  # floats


@pytest.mark.parametrize("n", [LARGE - 1, LARGE, LARGE + 1, 7 * SLOT, 8 * SLOT, 9 * SLOT + 3, 20 * SLOT - 1])
def test_large_reads(n):
    a, b = K.open("hip"), K.open("hip")
    x = np.random.default_rng(n).standard_normal(n, dtype=np.float32)
    xa, xb = a.upload(x), b.upload(-x)
    for _ in range(2):  # the barrier covers the work before the read; the ring is used again
        a.add_in_place(xa, xa, n)
        x = x + x
        assert np.array_equal(a.read(xa, n), x)
        assert np.array_equal(a.read(xa, n - 7), x[:n - 7])
    assert np.array_equal(b.read(xb, n), -np.random.default_rng(n).standard_normal(n, dtype=np.float32))
    a.close()
    b.close()
