"""Exact-grid products under graph capture: one call of the largest size on the
stream beforehand, on the matrix cores, then a call of that size that takes the
two-pass kernels (its output is its input) is captured and replayed.

Replays against the eager call: the same kernels on the same inputs, so the
same bits.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npt,M", [(700, 24), (2048, 70)])
def test_in_place_call_captured_after_a_matrix_core_warm_up(npt, M):
    from sfemans_amd import fft_parallele as FP
    from sfemans_amd._lib import check, lib
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    rng = np.random.default_rng(M)
    decay = np.exp(-np.arange(M) / 4.0)
    V = [rng.standard_normal((npt, 6, M)) * decay for _ in range(2)]
    s = rng.standard_normal((npt, 2, M)) * decay * 0.05
    s[:, 0, 0] = 1.5
    new = FP.fortran_empty
    Vd, sd = [FP.fortran_tensor(v) for v in V], FP.fortran_tensor(s)
    want = []
    for v in Vd:
        x = FP.fortran_tensor(np.zeros((npt, 6, M))).copy_(v)
        want.append(FP.FFT_SCALAR_VECT_DCL(None, x, sd, x, 2))
    got, out = new((npt, 6, M)), new((npt, 6, M))
    big = []                                                 # larger calls, on the matrix cores
    for n in (6000, 9000):
        x, y = torch.ones((32, 6, n), dtype=torch.float64, device="cuda"), torch.zeros((32, 2, n), dtype=torch.float64, device="cuda")
        y[0, 0] = 2.0
        big.append((x.permute(2, 1, 0), y.permute(2, 1, 0), new((n, 6, 32))))
    torch.cuda.synchronize()
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        FP.FFT_SCALAR_VECT_DCL(None, Vd[0], sd, out, 2)      # separate arrays
    st.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        FP.FFT_SCALAR_VECT_DCL(None, got, sd, got, 2)
    for i in (0, 1, 0):
        with torch.cuda.stream(st):                          # they reserve more scratch; the graph's stays
            FP.FFT_SCALAR_VECT_DCL(None, *big[i], 2)
        st.synchronize()
        got.copy_(Vd[i])
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want[i])
    del g
    check(lib().sfx_stream_release(st.cuda_stream))
