"""The matrix-core exact-grid kernel (sfx_exact_mm_body.h) on the CPU emulator
against the two-pass kernels and the oracle (CPU only).

Both evaluate the same sums of at most M and m_max_pad terms in another order:
their relative max-norm distance is below 4 (M + m_max_pad) eps times the
operation's amplification, bounded here by 1e-12 as everywhere in this suite.
"""
import numpy as np
import pytest

from oracle import fft_par as F
from tests import emu_runner

(EX_DIV, EX_SV2, EX_SQRT, EX_HEAVI, EX_TENSION, _, EX_SVCLAMP, EX_CLAMP01, EX_ENTRO, EX_GRADMOM, EX_COMPR) = range(11)
EX_CLS, EX_ETA, EX_ETA3, EX_FROMREAL = 13, 17, 18, 19


def rel(a, b):
    return np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300)


def both(op, npt, M, mp, in1, in2, out, values=None, eps=0.0, nb=2):
    vals = None if values is None else np.asarray(values, dtype=np.float64)
    res = []
    for fn in ("emu_exact", "emu_exact_mm"):
        rc, arrs = emu_runner.call(fn, op, npt, M, mp, in1, in2, vals, 0 if vals is None else len(vals), eps, nb,
                                   out.copy(order="K"))
        assert rc == 0
        res.append(arrs[-1])
    return res


def field(rng, npt, nb, M, scale=1.0, mean=None):
    V = rng.standard_normal((npt, nb, M)) * scale * np.exp(-np.arange(M) / 4.0)
    if mean is not None:
        V[:, 0, 0] = mean
    return np.asfortranarray(V)


def zeros(*shape):
    return np.zeros(shape, order="F")


# whole, ragged and short tiles; mode blocks 1 to 4 and two halves of 3; angle blocks 1, 2, 3,
# 5, 6, and more than one pass
SIZES = [(16, 4, 6), (33, 6, 17), (17, 16, 16), (5, 23, 34), (3, 48, 72), (2, 64, 96), (3, 17, 60), (2, 70, 105)]


@pytest.mark.parametrize("npt,M,mp", SIZES)
@pytest.mark.parametrize("op", [EX_DIV, EX_SV2, EX_TENSION, EX_ENTRO, EX_GRADMOM, EX_COMPR, EX_ETA3, EX_FROMREAL])
def test_against_two_pass(op, npt, M, mp):
    rng = np.random.default_rng(op * 100 + M)
    N = 2 * mp - 1
    flat = lambda *xs: np.concatenate([np.asarray(x).ravel(order="F") for x in xs])
    V, W, X = (field(rng, npt, 6, M) for _ in range(3))
    c = field(rng, npt, 2, M, 0.1, 1.5)
    creal = rng.random((N, npt))
    in1, in2, out, vals = {
        EX_DIV: (c, field(rng, npt, 2, M, 0.1, 2.0), zeros(npt, 2, M), None),
        EX_SV2: (V, c, zeros(npt, 6, M), None),
        EX_TENSION: (V, W, zeros(3, npt, 6, M), None),
        EX_ENTRO: (V, flat(c, creal), np.zeros(npt * 8 * M), [0.3]),
        EX_GRADMOM: (flat(V, W, X, creal), None, zeros(3, npt, 6, M), [0.2]),
        EX_COMPR: (flat(V, W), flat(c, creal), np.zeros(npt * 8 * M), [0.3, 1.5]),
        EX_ETA3: (V, np.asfortranarray(creal), zeros(npt, 6, M), None),
        EX_FROMREAL: (None, np.asfortranarray(creal), zeros(npt, 2, M), None),
    }[op]
    a, b = both(op, npt, M, mp, in1, in2, out, vals, nb=6 if op == EX_ETA3 else 2)
    assert rel(b, a) <= 1e-12


@pytest.mark.parametrize("pb", [1, 2])
def test_clamped_scalar(pb):
    rng = np.random.default_rng(pb)
    V, s = field(rng, 7, 6, 20), field(rng, 7, 2, 20, 0.4, 1.0)
    a, b = both(EX_SVCLAMP, 7, 20, 30, V, s, zeros(7, 6, 20), [0.6, 1.3], nb=pb)
    assert rel(b, a) <= 1e-12


@pytest.mark.parametrize("op,nb", [(EX_SQRT, 4), (EX_CLAMP01, 2), (EX_ETA, 2), (EX_CLS, 2)])
def test_scalar_ops(op, nb):
    rng = np.random.default_rng(op)
    npt, M, mp = 18, 9, 13
    c = field(rng, npt, nb, M, 0.3, 0.5)
    if op == EX_ETA:
        in1, in2, out, vals = c, np.asfortranarray(rng.random((2 * mp - 1, npt))), zeros(npt, 2, M), None
    elif op == EX_CLS:
        in1 = np.concatenate([field(rng, npt, 6, M).ravel(order="F"), field(rng, npt, 6, M, 0.1).ravel(order="F")])
        in2, out, vals = c, zeros(npt, 2, M), [1.0, 0.5, 0.05]
    else:
        in1, in2, out, vals = c, None, c, None
    a, b = both(op, npt, M, mp, in1, in2, out, vals, nb=nb)
    assert rel(b, a) <= 1e-12


@pytest.mark.parametrize("n_int", [1, 2, 3, 4])
def test_heaviside(n_int):
    rng = np.random.default_rng(n_int)
    V = rng.standard_normal((n_int, 5, 2, 12)) * 0.2
    V[:, :, 0, 0] += 0.5
    a, b = both(EX_HEAVI, 5, 12, 18, np.asfortranarray(V), None, zeros(5, 2, 12), list(np.linspace(1, 3, n_int + 1)), 0.2)
    assert rel(b, a) <= 1e-12


def test_nonfinite_stay_in_their_point():
    # an infinite coefficient, and a zero divisor whose quotients are not finite: other points are not touched
    rng = np.random.default_rng(3)
    c1, c2 = field(rng, 20, 2, 8), field(rng, 20, 2, 8, 0.05, 2.0)
    c1[3, 0, 2] = np.inf
    c2[17] = 0.0
    a, b = both(EX_DIV, 20, 8, 12, c1, c2, zeros(20, 2, 8))
    bad = [3, 17]
    good = [p for p in range(20) if p not in bad]
    assert rel(b[good], a[good]) <= 1e-12
    assert not np.isfinite(b[bad, 0, 0]).any() and not np.isfinite(a[bad, 0, 0]).any()
    c1[3, 0, 2], c2[17, 0, 0] = 0.0, 1.0
    c1[:, 1, 0], c2[:, 1, 0] = np.inf, np.nan      # the sine of mode 0 is not read
    a, b = both(EX_DIV, 20, 8, 12, c1, c2, zeros(20, 2, 8))
    assert np.isfinite(b).all() and rel(b, a) <= 1e-12


@pytest.mark.parametrize("me,lg,M,mp", [(5, 7, 6, 9), (7, 3, 20, 30)])
def test_entropy_visc(me, lg, M, mp):
    rng = np.random.default_rng(me)
    npt = me * lg
    V = [field(rng, npt, 6, M) for _ in range(5)]
    h = rng.random(npt) * 0.1
    out = np.zeros(3 * npt * 6 * M)
    rc, arrs = emu_runner.call("emu_exact_evisc_mm", npt, M, mp, lg, np.concatenate([v.ravel(order="F") for v in V]), h,
                               0.3, 0.9, 0.8, 1.0, out)
    assert rc == 0
    got = arrs[-1].reshape(3, -1)
    ref = F.fft_compute_entropy_visc(*V, h, 1.0, lg, 0.3, 0.9, 0.8, mp)
    for g, r in zip(got, ref):
        assert rel(g, np.asarray(r).ravel(order="F")) <= 1e-12
