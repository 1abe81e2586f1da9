"""Exact-grid products at the sizes where the route changes (exact_mm_use) and at
the edges of the matrix-core kernel's tiles, against the oracle.

Relative max-norm error <= 1e-12: sums of at most 128 + 192 terms of order one
and a pointwise operation with derivatives of order one, in double precision.
"""
import numpy as np
import pytest

from oracle import fft_par as F

pytestmark = pytest.mark.gpu

# (points, M, m_max_pad): tiles of 16 points (15, 16, 17), mode blocks 1-4 whole and ragged, both
# exact forms (jbn = JB and JB - 1), a wide grid, more than 64 modes below and above 2,048 points,
# few modes below and above 16,384 points
SIZES = [(15, 16, 24), (16, 32, 48), (17, 33, 49), (40, 64, 96), (31, 47, 70), (33, 57, 85), (37, 17, 60),
         (50, 1, 1), (2048, 80, 120), (2049, 80, 120), (9, 128, 192), (16384, 4, 6), (16385, 4, 6), (16385, 8, 12)]


def rel(t, ref):
    return np.max(np.abs(t.cpu().numpy() - ref)) / np.max(np.abs(ref))


def field(rng, npt, nb, M, scale=1.0, mean=None):
    V = rng.standard_normal((npt, nb, M)) * scale * np.exp(-np.arange(M) / 4.0)
    if mean is not None:
        V[:, 0, 0] = mean
    return np.asfortranarray(V)


@pytest.mark.parametrize("npt,M,mp", SIZES)
def test_products(npt, M, mp):
    import torch
    from sfemans_amd import fft_parallele as FP
    rng = np.random.default_rng(1000 * M + npt)
    dev, new = FP.fortran_tensor, FP.fortran_empty
    V, W, c, d = field(rng, npt, 6, M), field(rng, npt, 6, M), field(rng, npt, 2, M), field(rng, npt, 2, M, 0.05, 1.5)
    eta = np.asfortranarray(rng.random((2 * mp - 1, npt)) + 0.5)
    o2, o6, o3 = new((npt, 2, M)), new((npt, 6, M)), new((3, npt, 6, M))
    FP.FFT_PAR_DIV_DCL(None, dev(c), dev(d), o2, m_max_pad=mp)
    assert rel(o2, F.fft_par_div_dcl(c, d, mp)) <= 1e-12
    FP.FFT_SCALAR_VECT_DCL(None, dev(V), dev(d), o6, 2, m_max_pad=mp)
    assert rel(o6, F.fft_scalar_vect_dcl(V, d, 2, mp)) <= 1e-12
    FP.FFT_PAR_VAR_ETA_PROD_T_DCL(None, dev(eta), None, dev(V), o6, m_max_pad=mp)
    assert rel(o6, F.fft_par_var_eta_prod(eta, V, mp)) <= 1e-12
    FP.FFT_TENSOR_DCL(None, dev(V), dev(W), o3, m_max_pad=mp, opt_tension=True)
    assert rel(o3, F.fft_tensor_dcl(V, W, mp, opt_tension=True)) <= 1e-12
    torch.cuda.synchronize()


@pytest.mark.parametrize("npt,M", [(700, 24), (700, 64)])
def test_output_over_input(npt, M):
    # an output array that is one of the inputs: every input is read before the first store
    from sfemans_amd import fft_parallele as FP
    rng = np.random.default_rng(M)
    V, W, d = field(rng, npt, 6, M), field(rng, npt, 6, M), field(rng, npt, 2, M, 0.05, 1.5)
    dev, new = FP.fortran_tensor, FP.fortran_empty
    ref, got = new((npt, 6, M)), dev(V)
    FP.FFT_SCALAR_VECT_DCL(None, dev(V), dev(d), ref, 2)
    FP.FFT_SCALAR_VECT_DCL(None, got, dev(d), got, 2)
    assert rel(got, ref.cpu().numpy()) <= 1e-12
    # entropy viscosity whose outputs are its tensor rows, in another order
    lg, h = 7, np.full(npt, 0.01)
    u, r = dev(V), dev(W)
    rows = [field(rng, npt, 6, M) for _ in range(3)]
    refs = [new((npt, 6, M)) for _ in range(3)]
    g = [dev(x) for x in rows]
    args = (1.0, lg, 0.3, 0.9, 0.8)
    hd = FP.fortran_tensor(h)
    FP.FFT_COMPUTE_ENTROPY_VISC(None, None, u, r, *[dev(x) for x in rows], hd, *refs, *args)
    FP.FFT_COMPUTE_ENTROPY_VISC(None, None, u, r, *g, hd, g[1], g[2], g[0], *args)
    for a, b in zip((g[1], g[2], g[0]), refs):
        assert rel(a, b.cpu().numpy()) <= 1e-12
