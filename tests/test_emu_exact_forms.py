"""The entropy-viscosity form of the matrix-core kernel on the CPU emulator at
sizes with angle blocks that are neither the first nor the last (they read the
neighbouring angles without a wrap), and in more than one pass over the angles,
against the oracle (bounds checked; CPU only).  Tolerance as in
test_emu_exact_mm.py.
"""
import numpy as np
import pytest

from oracle import fft_par as F
from tests import emu_runner
from tests.test_emu_exact_mm import field, rel


# (elements, points per element, modes, m_max_pad): 3 and 7 angle blocks, of one and of two mode blocks; more than 64 modes
@pytest.mark.parametrize("me,lg,M,mp", [(2, 7, 20, 40), (5, 7, 6, 100), (3, 7, 70, 105), (1, 3, 128, 192)])
def test_entropy_visc(me, lg, M, mp):
    rng = np.random.default_rng(me + M)
    npt = me * lg
    V = [field(rng, npt, 6, M) for _ in range(5)]
    h = rng.random(npt) * 0.1
    out = np.zeros(3 * npt * 6 * M)
    rc, arrs = emu_runner.call("emu_exact_evisc_mm", npt, M, mp, lg, np.concatenate([v.ravel(order="F") for v in V]), h,
                               0.3, 0.9, 0.8, 1.0, out)
    assert rc == 0
    ref = F.fft_compute_entropy_visc(*V, h, 1.0, lg, 0.3, 0.9, 0.8, mp)
    for g, r in zip(arrs[-1].reshape(3, -1), ref):
        assert rel(g, np.asarray(r).ravel(order="F")) <= 1e-12
