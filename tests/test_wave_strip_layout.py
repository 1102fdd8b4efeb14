"""The LDS strips of the wave-strip backprojector, on the host: every wave's strip starts
at a multiple of 16 bytes, which its 16-byte stores need, and holds the run's columns
before its zero slot."""
import ctypes
import math

import pytest

from launch_rules import rules


@pytest.mark.parametrize("sides", [1, 2])
@pytest.mark.parametrize("zpt", [1, 2, 4, 8])
def test_strips_are_aligned(sides, zpt):
    columns = rules().check_wave_strip_columns
    columns.argtypes = [ctypes.c_double, ctypes.c_int, ctypes.c_int]
    for k in range(1, 400):
        dvz = 0.01 * k
        ct = columns(dvz, zpt, sides)
        for wave in range(4):
            assert wave * ct * sides * 4 % 16 == 0, (dvz, ct, wave)
        # span, one tap more, and up to 3 columns before it, in whole quads
        quads = math.ceil((math.ceil(dvz * (64 * zpt - 1)) + 2 + 3) / 4)
        assert 4 * quads <= ct - 2
    assert columns(1e9, zpt, sides) == 0
