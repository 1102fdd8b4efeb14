"""When 16-bit views with odd rows are copied for the wave-strip backprojector, against
the times measured both ways (microseconds: gather kernel, copy): the rule never takes
the slower way by more than a microsecond or two, and never copies a single view."""
import ctypes

import pytest

from launch_rules import rules

# n (volume n^3, views (n + 1)^2), slabs, views: gather, copy
MEASURED = {
    (48, 2, 32): (68.1, 28.0), (48, 1, 32): (36.3, 19.2), (64, 2, 32): (67.9, 38.0),
    (64, 1, 32): (35.9, 23.4), (80, 2, 8): (36.1, 23.7), (80, 2, 32): (128.9, 48.9),
    (96, 2, 4): (20.3, 22.4), (96, 2, 8): (36.8, 27.9), (96, 1, 4): (11.9, 17.9),
    (128, 2, 4): (31.1, 28.4), (128, 2, 8): (57.6, 39.9), (160, 2, 1): (17.6, 29.5),
    (160, 1, 1): (11.6, 20.7), (160, 2, 2): (27.7, 30.6), (160, 1, 2): (16.6, 22.8),
    (160, 1, 3): (21.6, 24.7), (200, 2, 1): (36.2, 41.8), (200, 1, 1): (22.5, 28.1),
    (200, 2, 4): (99.9, 56.8), (256, 2, 1): (48.7, 60.9), (256, 1, 1): (31.0, 41.4),
    (256, 2, 4): (133.9, 84.9), (256, 1, 32): (463.0, 211.1), (400, 2, 1): (143.3, 171.0),
    (400, 1, 1): (137.0, 150.3), (512, 1, 1): (391.4, 428.0), (512, 2, 32): (3947.5, 1652.9),
}


def pays(n, slabs, views):
    fn = rules().check_pitched_copy_pays
    fn.argtypes = [ctypes.c_double, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_double]
    return bool(fn(n * n, n // slabs, slabs, views, (n + 4) // 4 * 4 * (n + 1)))


@pytest.mark.parametrize("case", list(MEASURED))
def test_measured_sizes(case):
    gather, copy = MEASURED[case]
    taken = copy if pays(*case) else gather
    assert taken <= min(gather, copy) + 2.0, (case, taken)


@pytest.mark.parametrize("n", [16, 100, 512, 2000])
def test_one_view_is_never_copied(n):
    assert not pays(n, 1, 1) and not pays(n, 2, 1)
