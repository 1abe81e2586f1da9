"""Every exact-grid product on the forms that the other GPU tests reach for a few
of them only: the two-pass kernels (more than 64 modes on more than 2,048 points)
and the general form of the matrix-core kernel (more than 64 modes, or a wider
grid, on few points), against the oracle; and the two-pass scratch of two
streams at once.

Relative max-norm error <= 1e-12 as in test_gpu_exact.py: sums of at most 128 + 192
terms of order one and a pointwise operation with derivatives of order one,
in double precision.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from oracle import fft_par as F  # noqa: E402
from sfemans_amd import fft_parallele as FP  # noqa: E402
from sfemans_amd._lib import check, lib  # noqa: E402

TOL = 1e-12
# (points, modes, m_max_pad): two passes; the general form: two parts of the modes, a wide grid, the largest
SIZES = [(2051, 80, 120), (35, 70, 105), (42, 20, 100), (14, 128, 192)]


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    yield


def near(t, ref):
    ref = np.asarray(ref)
    return np.max(np.abs(t.cpu().numpy() - ref)) <= TOL * np.max(np.abs(ref))


def fields(rng, npt, nb, M, scale=1.0, mean=None):
    V = rng.standard_normal((npt, nb, M)) * scale * np.exp(-np.arange(M) / 4.0)
    if mean is not None:
        V[:, 0, 0] = mean
    return np.asfortranarray(V)


dev, new = FP.fortran_tensor, FP.fortran_empty


@pytest.mark.parametrize("npt,M,mp", SIZES)
@pytest.mark.parametrize("n_int", [1, 2, 3, 4])
def test_heaviside(npt, M, mp, n_int):
    rng = np.random.default_rng(10 * M + n_int)
    V = rng.standard_normal((n_int, npt, 2, M)) * 0.3 * np.exp(-np.arange(M) / 3.0)
    V[:, :, 0, 0] += 0.5
    vals, out = np.linspace(1.0, 5.0, n_int + 1), new((npt, 2, M))
    FP.FFT_HEAVISIDE_DCL(None, dev(V), vals, out, m_max_pad=mp, coeff_tanh=0.2)
    assert near(out, F.fft_heaviside_dcl(V, vals, mp, 0.2))


@pytest.mark.parametrize("npt,M,mp", SIZES)
def test_scalar_products(npt, M, mp):
    rng = np.random.default_rng(20 + M)
    c, V, W = fields(rng, npt, 4, M, 0.4, 0.5), fields(rng, npt, 6, M), fields(rng, npt, 6, M)
    for call, ref in ((FP.FFT_SQUAREROOT_SCALAR, F.fft_squareroot_scalar),
                      (FP.FFT_NO_OVERSHOOT_LEVEL_SET, F.fft_no_overshoot_level_set)):
        exp = c.copy()
        exp[:, 0:2] = ref(c, mp)
        d = dev(c)
        call(None, d, m_max_pad=mp)
        assert near(d, exp)
    s, bounds, o6, o2 = fields(rng, npt, 2, M, 0.4, 1.5), np.array([1.2, 1.8]), new((npt, 6, M)), new((npt, 2, M))
    for pb in (1, 2):
        FP.FFT_SCALAR_VECT_NO_OVERSHOOT(None, bounds, dev(V), dev(s), o6, pb, m_max_pad=mp)
        assert near(o6, F.fft_scalar_vect_no_overshoot(bounds, V, s, pb, mp))
    c = np.asfortranarray(c[:, :2])
    vals = (1.3, 0.7, 0.05)
    FP.FFT_COMPRESSION_LEVEL_SET_DCL(None, None, dev(V), dev(W), dev(c), o2, None, 7, *vals, m_max_pad=mp)
    assert near(o2, F.fft_compression_level_set_dcl(V, W, c, 7, *vals, mp))


@pytest.mark.parametrize("npt,M,mp", SIZES)
def test_entropy_viscosities(npt, M, mp):
    rng = np.random.default_rng(30 + M)
    V = [fields(rng, npt, 6, M) for _ in range(5)]
    c = fields(rng, npt, 2, M, 0.3, 0.5)
    creal = np.asfortranarray(rng.standard_normal((2 * mp - 1, npt)))
    o6, o2, o3 = new((npt, 6, M)), new((npt, 2, M)), new((3, npt, 6, M))
    FP.FFT_PAR_ENTRO_VISC_DCL(None, dev(V[0]), dev(c), dev(creal), None, 0.3, o6, o2, m_max_pad=mp)
    for o, r in zip((o6, o2), F.fft_par_entro_visc_dcl(V[0], c, creal, 0.3, mp)):
        assert near(o, r)
    FP.FFT_PAR_COMPR_ENTRO_VISC_DCL(None, dev(V[0]), dev(V[1]), dev(c), dev(creal), None, 0.3, o6, o2, 1.7, m_max_pad=mp)
    for o, r in zip((o6, o2), F.fft_par_compr_entro_visc_dcl(V[0], V[1], c, creal, 0.3, 1.7, mp)):
        assert near(o, r)
    FP.FFT_COMPUTE_ENTROPY_VISC_GRAD_MOM(None, *[dev(v) for v in V[:3]], dev(creal), o3, 0.25, m_max_pad=mp)
    assert near(o3, F.fft_compute_entropy_visc_grad_mom(*V[:3], creal, 0.25, mp))
    h, outs = rng.uniform(0.1, 1.0, npt), [new((npt, 6, M)) for _ in range(3)]
    FP.FFT_COMPUTE_ENTROPY_VISC(None, None, *[dev(v) for v in V], dev(h), *outs, 1.7, 7, 0.3, 0.9, 0.8, m_max_pad=mp)
    for o, r in zip(outs, F.fft_compute_entropy_visc(*V, h, 1.7, 7, 0.3, 0.9, 0.8, mp)):
        assert near(o, r)


# few modes, on both sides of the lines of exact_mm_use: 2,400 elements of 7 points (two passes) and 600
@pytest.mark.parametrize("npt", [4200, 16800])
def test_few_modes(npt):
    M, mp = 2, 3
    rng = np.random.default_rng(npt)
    V, h = [fields(rng, npt, 6, M) for _ in range(5)], rng.uniform(0.1, 1.0, npt)
    outs, o3 = [new((npt, 6, M)) for _ in range(3)], new((3, npt, 6, M))
    FP.FFT_COMPUTE_ENTROPY_VISC(None, None, *[dev(v) for v in V], dev(h), *outs, 1.7, 7, 0.3, 0.9, 0.8)
    for o, r in zip(outs, F.fft_compute_entropy_visc(*V, h, 1.7, 7, 0.3, 0.9, 0.8, mp)):
        assert near(o, r)
    FP.FFT_TENSOR_DCL(None, dev(V[0]), dev(V[1]), o3, opt_tension=True)
    assert near(o3, F.fft_tensor_dcl(V[0], V[1], mp, opt_tension=True))


def test_two_streams_on_the_two_pass_kernels():
    # stream A grows its scratch between two calls while B divides; bit for bit the calls one after the other
    rng = np.random.default_rng(91)
    nA, nB, M = 6000, 5000, 72
    V, c = [dev(fields(rng, nA, 6, M)) for _ in range(2)], [fields(rng, nB, 2, M), fields(rng, nB, 2, M, 0.1, 2.0)]
    small, c = [dev(np.asfortranarray(x[:2100])) for x in c], [dev(x) for x in c]
    torch.cuda.synchronize()

    def tension(o):
        return FP.FFT_TENSOR_DCL(None, *V, o, opt_tension=True)

    refT = tension(new((3, nA, 6, M)))
    refS, refD = FP.FFT_PAR_DIV_DCL(None, *small, new((2100, 2, M))), FP.FFT_PAR_DIV_DCL(None, *c, new((nB, 2, M)))
    T, S, D = ([new(s) for _ in range(3)] for s in ((3, nA, 6, M), (2100, 2, M), (nB, 2, M)))
    torch.cuda.synchronize()
    sA, sB = torch.cuda.Stream(), torch.cuda.Stream()
    try:
        for i in range(3):
            with torch.cuda.stream(sA):
                FP.FFT_PAR_DIV_DCL(None, *small, S[i])
                tension(T[i])
            with torch.cuda.stream(sB):
                FP.FFT_PAR_DIV_DCL(None, *c, D[i])
        torch.cuda.synchronize()
    finally:
        check(lib().sfx_stream_release(sA.cuda_stream))
        check(lib().sfx_stream_release(sB.cuda_stream))
    for o, r in ((T, refT), (S, refS), (D, refD)):
        assert all(torch.equal(x, r) for x in o)
