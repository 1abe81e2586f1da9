"""Results of the host-pointer entry points on their way to the caller
(sfx_hostcopy.cpp) on a HIP runtime in host memory (CPU only): which copies
take the page-locked ring, what it holds when it is kept, two threads, errors.
The fake runtime runs an asynchronous copy only when an event behind it or its
stream is waited for, so a chunk that is read too early is not there yet.
"""
import numpy as np
import pytest

from tests import host_runner

pytestmark = pytest.mark.skipif(host_runner.hipcc() is None, reason="hipcc not found")

MB = 1 << 20
MIN, MAX = 2 * MB, 32 * MB     # shortest and longest copy through the ring


@pytest.fixture
def L():
    return host_runner.load()


def copy(L, n, seed):
    src = np.random.default_rng(seed).integers(0, 256, n + 16, dtype=np.uint8)
    dst = np.full(n + 16, 0xA5, dtype=np.uint8)
    rc = L.host_copy_out(dst.ctypes.data, src.ctypes.data, n)
    return rc, np.array_equal(dst[:n], src[:n]) and (dst[n:] == 0xA5).all()


def routes(L):
    r = L.fake_count(b"memcpy"), L.fake_count(b"copy")
    L.fake_reset_counts()
    return r


@pytest.mark.parametrize("n,chunks", [(MIN - 1, 0), (MIN, 2), (MIN + 1, 3), (4 * MB, 4), (5 * MB + 8, 6), (MAX, 32),
                                      (MAX + 1, 0)])
def test_route_and_bytes(L, n, chunks):
    assert copy(L, n, n) == (0, True)
    assert routes(L) == ((0, chunks) if chunks else (1, 0))
    assert L.fake_pending() == 0


def test_kept_ring(L):
    # one ring for copies of other data and other lengths, long and short in turn
    for i, n in enumerate((9 * MB + 3, MIN, 6 * MB, MIN + 5, 13 * MB)):
        assert copy(L, n, i) == (0, True)
        assert L.fake_count(b"memcpy") == 0
    assert L.fake_count(b"hostmalloc") == 1 and L.fake_count(b"event") == 4
    # given back with the null stream's scratch, made again by the next copy
    assert L.sfx_stream_release(None) == 0 and L.fake_count(b"hostfree") == 1
    assert copy(L, 3 * MB, 9) == (0, True) and L.fake_count(b"hostmalloc") == 2


def test_pinned_memory_and_no_ring_take_memcpy(L):
    src, dst = np.arange(3 * MB, dtype=np.uint8), np.zeros(3 * MB, dtype=np.uint8)
    L.fake_pin(dst.ctypes.data, 1)
    assert L.host_copy_out(dst.ctypes.data, src.ctypes.data, dst.nbytes) == 0 and np.array_equal(src, dst)
    L.fake_pin(dst.ctypes.data, 0)
    assert routes(L) == (1, 0)
    L.fake_limit(MB)                      # no page-locked memory to be had
    assert copy(L, 3 * MB, 1) == (0, True) and routes(L) == (1, 0)
    assert L.fake_last_error() == 0
    L.fake_limit(0)
    assert copy(L, 3 * MB, 1) == (0, True) and routes(L) == (0, 3)


def test_a_second_thread_takes_memcpy(L):
    src = np.random.default_rng(0).integers(0, 256, 4 * MB, dtype=np.uint8)
    dst = np.zeros_like(src)
    L.host_copy_out_meanwhile(dst.ctypes.data, src.ctypes.data, src.nbytes)
    assert copy(L, 7 * MB, 2) == (0, True)
    assert L.host_copy_out_meanwhile_rc() == 0 and np.array_equal(src, dst)
    assert routes(L) == (1, 7)


@pytest.mark.parametrize("copies,records", [(0, -1), (3, -1), (6, -1), (-1, 0), (-1, 5)])
def test_error_leaves_no_copy_under_way(L, copies, records):
    L.fake_fail(copies, records)
    rc, _ = copy(L, 8 * MB, 3)
    assert rc != 0 and L.fake_pending() == 0
    L.fake_fail(-1, -1)
    assert copy(L, 8 * MB, 4) == (0, True)
