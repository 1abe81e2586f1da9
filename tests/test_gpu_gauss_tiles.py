"""Tilings of the fused Gauss-point kernels vs the oracle: sizes on both sides
of the rule between whole elements and point tiles, and half tiles whose last
work-group is partly or wholly past an odd number of elements.

Tolerance: relative max-norm error <= 1e-12 (FP64), as for the kernels' other
sizes; the element sums against their two-step form, 1e-12.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from oracle import smb  # noqa: E402
from sfemans_amd import nonlinear as NL  # noqa: E402
from sfemans_amd.fft_parallele import fortran_empty, fortran_tensor  # noqa: E402
from sfemans_amd.mesh import P2Mesh, rectangle_p2  # noqa: E402
from sfemans_amd.synth import fourier_field  # noqa: E402

TOL = 1e-12


def rel(a, b):
    return np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300)


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    yield


def odd_mesh(nx, ny):
    """The rectangle without its last triangle (and the nodes that it alone has)."""
    m = rectangle_p2(nx, ny)
    jj = m.jj[:, :-1]
    used, inv = np.unique(jj, return_inverse=True)
    return P2Mesh((inv.reshape(jj.shape) + 1).astype(np.int32), m.rr[:, used - 1])


# work-groups of whole elements / of points: (169, 296), (150, 263) and (180, 315)
# take whole elements, (146, 256), (125, 219) and (100, 175) point tiles, as do
# (282, 493) and (300, 525)
@pytest.mark.parametrize("nx,ny,M", [(60, 90, 3), (40, 60, 8), (12, 15, 100), (60, 78, 3), (40, 50, 8), (10, 10, 100),
                                     (95, 95, 4), (15, 20, 70)])
def test_whole_elements_or_points(nx, ny, M):
    print(f"case tiles cross_curl {nx}x{ny} M={M}", flush=True)
    m = rectangle_p2(nx, ny)
    modes = np.arange(M)
    u = fourier_field(m.np, 6, M, 21, 2.0)
    out = np.zeros((m.n_gauss, 6, M), order="F")
    NL.smb_cross_prod_gauss_sft_par(None, NL.Mesh.from_p2(m), modes, u, out)
    assert rel(out, smb.smb_cross_prod_gauss_sft_par(m.jj, m.rr, modes, u)) <= TOL


@pytest.mark.parametrize("M", [3, 5, 13, 24, 64, 100])
def test_half_tiles_odd_elements(M):
    print(f"case tiles odd M={M}", flush=True)
    m = odd_mesh(5, 4) if M < 64 else odd_mesh(2, 3)
    mesh = NL.Mesh.from_p2(m)
    modes = np.arange(M)
    U, D = (fourier_field(m.np, 6, M, s, 2.0) for s in (22, 23))
    c = fourier_field(m.np, 2, M, 24, 2.0)
    hc = 0.5 + np.random.default_rng(25).random(m.me)
    G = 7 * m.me
    out = np.zeros((G, 6, M), order="F")
    NL.nl_tangent(mesh, modes, U, D, out)
    assert rel(out, smb.smb_CurlH_cross_B_gauss_sft_par(m.jj, m.rr, modes, U, D)
               + smb.smb_CurlH_cross_B_gauss_sft_par(m.jj, m.rr, modes, D, U)) <= TOL
    oc = np.zeros((G, 2, M), order="F")
    NL.smb_ugradc_gauss_fft_par(None, mesh, modes, hc, U, c, oc)
    assert rel(oc, smb.smb_ugradc_gauss_fft_par(m.jj, m.rr, modes, hc, U, c)) <= TOL
    # the fused right-hand side against the Gauss output and its assembly
    dU, g = fortran_tensor(U), fortran_empty((G, 6, M))
    one, two = ([fortran_empty((m.np, 3, M)) for _ in range(2)] for _ in range(2))
    NL.smb_cross_prod_gauss_sft_par(None, mesh, modes, dU, g)
    NL.nl_rhs_3x3(mesh, modes, dU, one[0], one[1], -1.0, None)
    NL.rhs_3x3_all_modes(mesh, g, two[0], two[1], -1.0)
    for a, b in zip(one, two):
        assert rel(a.cpu().numpy(), b.cpu().numpy()) <= TOL
    # <T d, y> = <d, T^T y>
    y, back, t = fortran_tensor(fourier_field(G, 6, M, 26, 2.0)), fortran_empty((m.np, 6, M)), fortran_empty((G, 6, M))
    NL.nl_adjoint(mesh, modes, dU, y, back)
    dD = fortran_tensor(D)
    NL.nl_tangent(mesh, modes, dU, dD, t)
    lhs, rhs = float((t * y).sum()), float((dD * back).sum())
    scale = float((t.abs() * y.abs()).sum())
    assert abs(lhs - rhs) <= TOL * scale
