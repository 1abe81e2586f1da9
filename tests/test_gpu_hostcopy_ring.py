"""Host-pointer results through a ring that is kept from one call to the next:
other data and other lengths each time, long ones and short ones in turn, one
result and three, against the device-pointer calls bit for bit.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def test_kept_ring_between_calls():
    from sfemans_amd import fft_parallele as FP
    from sfemans_amd._lib import check, lib
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    M = 2                              # 96 bytes of result per point
    check(lib().sfx_stream_release(None))
    for i, npt in enumerate((98308, 21847, 65541, 21000, 140007, 43694)):
        rng = np.random.default_rng(i)
        V = [np.asfortranarray(rng.standard_normal((npt, 6, M))) for _ in range(2)]
        out, dev = np.full((npt, 6, M), np.nan, order="F"), FP.fortran_empty((npt, 6, M))
        FP.FFT_PAR_CROSS_PROD_DCL(None, *V, out)
        FP.FFT_PAR_CROSS_PROD_DCL(None, *[FP.fortran_tensor(v) for v in V], dev)
        assert np.array_equal(out, dev.cpu().numpy()), npt
    npt = 7 * 7001                     # three results of 4.5 MB
    rng = np.random.default_rng(9)
    V = [np.asfortranarray(rng.standard_normal((npt, 6, M))) for _ in range(5)]
    h, args = np.full(npt, 0.01), (1.0, 7, 0.3, 0.9, 0.8)
    outs = [np.full((npt, 6, M), np.nan, order="F") for _ in range(3)]
    devs = [FP.fortran_empty((npt, 6, M)) for _ in range(3)]
    FP.FFT_COMPUTE_ENTROPY_VISC(None, None, *V, h, *outs, *args)
    FP.FFT_COMPUTE_ENTROPY_VISC(None, None, *[FP.fortran_tensor(v) for v in V], FP.fortran_tensor(h), *devs, *args)
    for o, d in zip(outs, devs):
        assert np.array_equal(o, d.cpu().numpy())
