"""Modes per work-group of the momentum right-hand side: few where eight would
leave most of the 256 CUs idle, eight elsewhere (CPU only; emu_rhs_ns runs both
forms and compares them bit for bit, see test_emu_rhs_tile.py for the sizes).
"""
import ctypes

import pytest

from tests import emu_runner


# (triangles, modes): 13 work-groups of eight modes, 208, 319; 320, and the sizes of a production run
@pytest.mark.parametrize("me,M,modes", [(400, 8, 2), (400, 128, 2), (32 * 319, 8, 2), (32 * 320, 8, 8), (102720, 48, 8),
                                        (200704, 1, 8), (10**7, 256, 8)])
def test_work_groups_fill_the_chip(me, M, modes):
    L = ctypes.CDLL(emu_runner.build_emulator())
    L.emu_rns_modes.argtypes = [ctypes.c_int64, ctypes.c_int]
    assert L.emu_rns_modes(me, M) == modes
