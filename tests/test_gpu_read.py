"""Reads on both sides of the size from which a read goes through pinned slots:
below it, one slot short of and past all of them, and a partial last slot; with
fewer slots and threads; and by several contexts at once."""

import threading

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


# no slot or no thread: one pageable copy; one slot for all pieces, more threads
# than slots, and one thread for all slots
@pytest.mark.parametrize("slots,threads", [(0, 8), (8, 0), (1, 1), (1, 3), (2, 8), (8, 1)])
def test_large_reads_with_less(slots, threads):
    n = 5 * SLOT + 3
    h = K.open("hip")
    h.dbg_read_limits(slots, threads)
    x = np.random.default_rng(n).standard_normal(n, dtype=np.float32)
    xb = h.upload(x)
    for _ in range(2):
        h.add_in_place(xb, xb, n)
        x = x + x
        assert np.array_equal(h.read(xb, n), x)
    h.close()


def test_large_reads_of_several_contexts():
    # the slots are shared by the process; contexts come and go meanwhile
    wrong = []

    def one(seed):
        x = np.random.default_rng(seed).standard_normal(3 * SLOT + seed, dtype=np.float32)
        for _ in range(4):
            h = K.open("hip")
            xb = h.upload(x)
            for _ in range(3):
                if not np.array_equal(h.read(xb, x.size), x):
                    wrong.append(seed)
            h.close()

    threads = [threading.Thread(target=one, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
