"""Scratch of the exact-grid products on the host side (CPU only, no GPU: a HIP
runtime in host memory).  The header's rule for graph capture: after one call
of the largest size on a stream, no call on it allocates, frees or waits,
whichever kernels it takes.
"""
import pytest

from tests import host_runner

pytestmark = pytest.mark.skipif(host_runner.hipcc() is None, reason="hipcc not found")

STREAM = 0x1000
A, B, S, O = (0x100000000000 + (i << 40) for i in range(4))   # arrays that do not overlap; never read


@pytest.fixture
def L():
    return host_runner.load()


def sv2(L, out, np_, M, v=A, mp=None, stream=STREAM):
    return L.sfx_fft_scalar_vect_dcl_dev(v, S, out, np_, M, 2, 3 * M // 2 if mp is None else mp, stream)


def routes(L):
    return L.fake_count(b"matrix"), L.fake_count(b"twopass")


# (warm-up, captured) as (np, M, in place): a call of the same size whose output is its input; more than
# 2,048 points of more than 64 modes; few modes on many points (smaller in scratch than the warm-up)
CASES = [((3000, 16, False), (3000, 16, True)), ((3000, 16, False), (2999, 16, True)),
         ((2048, 80, False), (2049, 79, False)), ((70000, 8, False), (60000, 4, False))]


@pytest.mark.parametrize("warm,cap", CASES)
def test_warm_up_is_enough_for_a_capture(L, warm, cap):
    for n, M, inplace in (warm, (8, cap[1], False)):       # the largest call, and the tables of the captured one
        assert sv2(L, A if inplace else O, n, M) == 0, L.sfx_last_error()
    assert routes(L)[1] == 0                               # all on the matrix cores
    L.fake_reset_counts()
    L.fake_capture(STREAM, 1)
    n, M, inplace = cap
    rc = sv2(L, A if inplace else O, n, M)
    broken = L.fake_capture_broken()
    L.fake_capture(None, 0)
    assert rc == 0 and not broken, L.sfx_last_error()
    assert routes(L) == (0, 1)
    assert [L.fake_count(k) for k in (b"malloc", b"free", b"sync")] == [0, 0, 0]


def test_no_reserve_inside_a_capture(L):
    # a matrix-core call larger than the warm-up needs no scratch: it is captured without any
    assert sv2(L, O, 1000, 16) == 0
    L.fake_reset_counts()
    L.fake_capture(STREAM, 1)
    rc = sv2(L, O, 5000, 16)
    broken = L.fake_capture_broken()
    L.fake_capture(None, 0)
    assert rc == 0 and not broken and routes(L) == (1, 0)
    assert L.fake_count(b"malloc") == 0 and L.fake_last_error() == 0


def test_another_stream_s_capture_is_left_alone(L):
    # first matrix-core call on a stream while another one is captured (its tables exist)
    assert sv2(L, O, 100, 16, stream=None) == 0
    L.fake_capture(0x2000, 1)
    rc = sv2(L, O, 1000, 16)
    broken = L.fake_capture_broken()
    L.fake_capture(None, 0)
    assert rc == 0 and not broken and routes(L)[0] == 2


def test_full_memory_does_not_refuse_a_matrix_core_call(L):
    assert sv2(L, O, 1000, 16) == 0
    used = L.fake_used()
    L.fake_limit(used + 1000)                              # no room for the larger scratch
    assert sv2(L, O, 5000, 16) == 0 and routes(L) == (2, 0)
    assert L.fake_last_error() == 0                        # left for no later check to find
    assert L.fake_used() == used                           # the smaller one is still there
    L.fake_capture(STREAM, 1)
    assert sv2(L, A, 1000, 16) == 0 and not L.fake_capture_broken()
    L.fake_capture(None, 0)
    assert sv2(L, A, 5000, 16) != 0                        # the two-pass call does need it


def test_null_stream_and_release(L):
    # the null stream cannot be captured: nothing is reserved for it beside the tables
    assert sv2(L, O, 1000, 16, stream=None) == 0
    tables = L.fake_used()
    assert sv2(L, O, 5000, 16, stream=None) == 0 and L.fake_used() == tables
    assert sv2(L, O, 5000, 16) == 0 and L.fake_used() == tables + 2 * 3 * 24 * 5000 * 8
    assert L.sfx_stream_release(STREAM) == 0 and L.fake_used() == tables


def test_a_captured_scratch_outlives_larger_matrix_core_calls(L):
    # a graph holds the scratch of an in-place call; larger calls on the matrix cores reserve more, and leave it
    assert sv2(L, A, 3000, 16) == 0
    L.fake_reset_counts()
    assert sv2(L, O, 5000, 16) == 0 and routes(L) == (1, 0)
    assert L.fake_count(b"free") == 0
    L.fake_capture(STREAM, 1)                              # and a larger in-place call can be captured after it
    rc = sv2(L, A, 5000, 16)
    broken = L.fake_capture_broken()
    L.fake_capture(None, 0)
    assert rc == 0 and not broken and L.fake_count(b"free") == 0


def test_scratch_is_bounded_and_given_back(L):
    assert sv2(L, O, 100, 16, stream=None) == 0
    tables = L.fake_used()
    for n in range(1000, 9000, 500):                       # growing calls on both kinds of kernels in turn
        assert sv2(L, A, n, 16) == 0 and sv2(L, O, n + 250, 16) == 0
        assert L.fake_used() - tables <= 2 * (2 * 3 * 24 * (n + 250) * 8)
    for n in range(10000, 20000, 1000):                    # on the matrix cores alone: one buffer
        assert sv2(L, O, n, 16) == 0
    assert L.sfx_stream_release(STREAM) == 0 and L.fake_used() == tables
