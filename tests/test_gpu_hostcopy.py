"""Results of the host-pointer entry points, copied back in page-locked chunks
of 1 MB (ring of 4): the same bytes as the device-pointer entry points write,
for results of less than two chunks or more than 32 (one hipMemcpy), of whole and of ragged
chunk counts, of more chunks than the ring has, and after the ring was given
back.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from sfemans_amd import fft_parallele as FP  # noqa: E402
from sfemans_amd._lib import check, lib  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    yield


# M = 2: 96 bytes of result per point, 2 MB at 21845.33 points
@pytest.mark.parametrize("npt", [21845, 21846, 32768, 43690, 43691, 54613, 54614, 98304, 120001, 349525, 349526])
@pytest.mark.parametrize("pinned", [False, True])
def test_host_result_is_the_device_result(npt, pinned):
    M = 2
    print(f"case hostcopy np={npt} pinned={pinned}", flush=True)
    rng = np.random.default_rng(npt)
    V1, V2 = (np.asfortranarray(rng.standard_normal((npt, 6, M))) for _ in range(2))
    d1, d2 = (torch.from_numpy(v.transpose(2, 1, 0).copy()).cuda().permute(2, 1, 0) for v in (V1, V2))
    dev = torch.zeros((M, 6, npt), dtype=torch.float64, device="cuda").permute(2, 1, 0)
    FP.FFT_PAR_CROSS_PROD_DCL(None, d1, d2, dev, 1, npt, 3 * M // 2)
    want = dev.cpu().numpy()
    for _ in range(2):
        out = torch.full((M, 6, npt), np.nan, dtype=torch.float64, pin_memory=pinned).numpy().transpose(2, 1, 0)
        FP.FFT_PAR_CROSS_PROD_DCL(None, V1, V2, out, 1, npt, 3 * M // 2)
        assert np.array_equal(out, want)
        check(lib().sfx_stream_release(None))
