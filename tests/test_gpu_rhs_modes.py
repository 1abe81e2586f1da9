"""The momentum right-hand side on both sides of the line between two and eight
modes per work-group: 200 tiles of elements, 16 modes (400 work-groups) in one
call against two calls of eight modes (200); 15 and 9 modes, ragged.

Relative max-norm distance <= 1e-13: the same sums of at most some 60 products
of order one in the same order, contracted to FMAs by the compiler in each form.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,tensor", [(16, False), (15, True), (9, False)])
def test_modes_together_and_apart(M, tensor):
    from sfemans_amd import nonlinear as NL
    from sfemans_amd.fft_parallele import fortran_empty, fortran_tensor
    from sfemans_amd.mesh import rectangle_p2
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    m = rectangle_p2(40, 80)
    mesh = NL.Mesh.from_p2(m)
    rng = np.random.default_rng(M)
    F = lambda *s: np.asfortranarray(rng.standard_normal(s))
    fields = [F(m.n_gauss, 6, M), F(m.np, 6, M), F(m.np, 6, M), F(m.np, 2, M), F(m.np, 2, M)]
    T = F(3, m.n_gauss, 6, M) if tensor else None

    def run(modes):
        part = [fortran_tensor(f[..., modes]) for f in fields]
        v = [fortran_empty((m.np, 3, len(modes))) for _ in range(2)]
        NL.rhs_ns_3x3(mesh, modes, *part, *v, opt_tensor=None if T is None else fortran_tensor(T[..., modes]))
        return [x.cpu().numpy() for x in v]

    whole = run(list(range(M)))
    first, rest = run(list(range(8))), run(list(range(8, M)))
    for w, a, b in zip(whole, first, rest):
        assert np.isfinite(w).all()
        assert np.max(np.abs(w - np.concatenate([a, b], axis=2))) <= 1e-13 * np.max(np.abs(w))
