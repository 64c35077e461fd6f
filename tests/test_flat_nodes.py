"""The flat D3Q27 launch's node mapping (lbm3d_step.hpp): every node once, in memory order."""
import ctypes
from pathlib import Path

import pytest

EMU = Path(__file__).resolve().parent / "emu" / "liblbm3d_emu.so"


@pytest.fixture(scope="module")
def emu():
    L = ctypes.CDLL(str(EMU))
    L.emu3_div_check.argtypes = [ctypes.c_uint32]
    return L


@pytest.mark.parametrize("shape", [(3, 3, 3), (250, 7, 5), (64, 64, 3), (65, 33, 9), (255, 3, 4), (257, 17, 3), (128, 128, 16)])
def test_flat_mapping_visits_every_node_once(emu, shape):
    assert emu.emu3_flat_check(*shape) == 0


@pytest.mark.parametrize("d", [2, 3, 5, 7, 63, 64, 65, 250, 1000, 4097, 65535, 65537, 1 << 20, (1 << 30) - 1, 1 << 30, (1 << 31) - 1])
def test_division_by_multiplication_is_exact(emu, d):
    assert emu.emu3_div_check(d) == 0
