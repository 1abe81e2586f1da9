"""Which kernels an exact-grid product takes (exact_mm_use), at sizes on both
sides of the lines where the other kernels were measured to be faster (CPU only:
the library's host code on a HIP runtime in host memory, launches recorded).
"""
import ctypes as C

import pytest

from tests import host_runner

pytestmark = pytest.mark.skipif(host_runner.hipcc() is None, reason="hipcc not found")

A = [0x100000000000 + (i << 40) for i in range(8)]     # arrays that do not overlap; never read
VALS = (C.c_double * 5)(1, 2, 3, 4, 5)


@pytest.fixture(scope="module")
def L():
    return host_runner.load()


def call(L, op, n, M):
    mp, i, i64, d, p = max(1, 3 * M // 2), C.c_int32, C.c_int64, C.c_double, C.c_void_p
    a = [p(x) for x in A]
    size = (i64(n), i(M))
    if op == "TENSION":
        rc = L.sfx_fft_tensor_dcl_dev(*a[:3], *size, i(mp), i(1), p(None))
    elif op == "COMPR":
        rc = L.sfx_fft_par_compr_entro_visc_dcl_dev(*a[:4], d(.3), d(1.), a[4], a[5], *size, i(mp), p(None))
    elif op == "EVISC":
        rc = L.sfx_fft_compute_entropy_visc_dev(*a[:5], a[5], a[6], a[7], p(A[7] + (1 << 39)), *size, i(mp), d(1.), i(7),
                                                d(.3), d(.9), d(.8), p(None))
    elif op == "CLS":
        rc = L.sfx_fft_compression_level_set_dcl_dev(*a[:4], *size, i(mp), d(1.), d(.5), d(.05), p(None))
    elif op.startswith("HEAVI"):
        rc = L.sfx_fft_heaviside_dcl_dev(a[0], VALS, a[1], i(int(op[5]) + 1), *size, i(mp), d(.2), p(None))
    elif op == "DIV":
        rc = L.sfx_fft_par_div_dcl_dev(*a[:3], *size, i(mp), p(None))
    elif op == "SV2":
        rc = L.sfx_fft_scalar_vect_dcl_dev(*a[:3], *size, i(2), i(mp), p(None))
    elif op == "GRADMOM":
        rc = L.sfx_fft_compute_entropy_visc_grad_mom_dev(*a[:4], d(.2), a[4], *size, i(mp), p(None))
    elif op == "ENTRO":
        rc = L.sfx_fft_par_entro_visc_dcl_dev(*a[:3], d(.3), a[3], a[4], *size, i(mp), p(None))
    elif op == "FROMREAL":
        rc = L.sfx_fft_par_from_real_dev(a[0], a[1], *size, i(mp), p(None))
    assert rc == 0, L.sfx_last_error()


# op, modes, (points, whether on the matrix cores)...
ROUTES = [("TENSION", 12, (16380, 1), (32767, 0), (131068, 1)), ("TENSION", 2, (8190, 1), (16380, 0), (262136, 0)),
          ("TENSION", 8, (16380, 1), (49140, 0)), ("TENSION", 16, (32767, 1), (131068, 1)),
          ("COMPR", 12, (8190, 1), (32767, 0), (131068, 0)), ("COMPR", 24, (8190, 1), (32767, 0), (131068, 1)),
          ("COMPR", 32, (32767, 1)), ("EVISC", 2, (8190, 1), (16380, 0)), ("EVISC", 6, (8190, 1), (65534, 0)),
          ("EVISC", 32, (351232, 1)), ("CLS", 17, (12285, 1), (131068, 0)), ("CLS", 64, (131068, 1)),
          ("HEAVI2", 24, (32767, 1), (131068, 0)), ("HEAVI2", 12, (131068, 1)), ("HEAVI4", 10, (49140, 1), (196602, 0)),
          ("DIV", 2, (65534, 1), (262136, 0)), ("SV2", 2, (32767, 1), (131068, 0)), ("SV2", 64, (402752, 1)),
          ("GRADMOM", 2, (16380, 1), (65534, 0)), ("ENTRO", 2, (32767, 1), (131068, 0)),
          ("FROMREAL", 1, (131068, 1), (402752, 0)), ("FROMREAL", 12, (402752, 1)),
          # the general form: more than 64 modes
          ("SV2", 80, (2048, 1), (2049, 0)), ("TENSION", 80, (2048, 1), (2049, 0))]


@pytest.mark.parametrize("route", ROUTES, ids=lambda r: f"{r[0]}-{r[1]}")
def test_route(L, route):
    op, M, *sizes = route
    for n, matrix in sizes:
        n -= n % 7 if op == "EVISC" else 0
        L.fake_reset_counts()
        call(L, op, n, M)
        want = (1, 0) if matrix else (0, 1)
        got = L.fake_count(b"matrix"), L.fake_count(b"twopass") - (op == "CLS")   # its maximum is a reduction
        assert got == want, (op, n)
