"""When single-slab runs of the wave-strip backprojector are taken instead of the older
kernels, against the times measured for both (microseconds: older kernel, runs).  Cubes of
n voxels of 256 / n mm, detectors n (samples a voxel) wide."""
import ctypes

import pytest

from launch_rules import rules

# n, slabs, samples a voxel step at unit magnification (detector / n), views: older, runs
MEASURED = {
    (256, 1, 1, 1): (37.6, 37.0), (256, 2, 1, 1): (41.8, 47.6), (160, 1, 1, 1): (11.5, 12.8),
    (160, 2, 1, 1): (17.8, 20.1), (128, 2, 1, 1): (11.1, 13.1), (300, 1, 1, 1): (64.4, 54.5), (400, 1, 1, 1): (148.4, 117.7),
    (512, 1, 1, 1): (343.9, 267.9), (640, 2, 1, 1): (886.3, 698.7), (640, 1, 1, 1): (744.0, 687.8),
    (512, 2, 1, 4): (671.7, 529.0), (512, 2, 1, 32): (3737.0, 1592.0), (512, 1, 1, 32): (3737.6, 1418.4),
    (400, 2, 1, 4): (322.6, 218.9), (400, 1, 1, 32): (2355.1, 785.8), (96, 2, 1, 2): (11.1, 9.4),
    (160, 1, 2, 4): (28.3, 38.8), (256, 1, 2, 4): (67.5, 126.1), (256, 1, 2, 32): (458.7, 544.7),
    (256, 1, 3, 4): (69.8, 126.4), (256, 1, 3, 32): (509.6, 552.8), (400, 2, 2, 4): (346.3, 617.6),
    (400, 1, 2, 4): (333.9, 541.1), (400, 2, 2, 32): (2417.9, 2774.7), (512, 2, 2, 32): (3800.4, 4588.7),
    (512, 1, 2, 32): (3797.2, 4589.3), (512, 1, 3, 4): (766.5, 1140.2), (512, 1, 3, 32): (3991.4, 4577.4),
}


def run(n, slabs, mult, views):
    fn = rules().check_wave_run
    fn.argtypes = [ctypes.c_double] + [ctypes.c_int] * 3 + [ctypes.POINTER(ctypes.c_int)]
    columns = ctypes.c_int()
    nearest = 1000 - 181 * (n - 1) / n  # the corner nearest to the source, in mm
    dvz = 256 / n * 1500 / nearest / (1.62 * 256 / (n * mult))
    return fn(dvz, n // slabs, 1, views, ctypes.byref(columns)), columns.value, dvz


@pytest.mark.parametrize("case", list(MEASURED))
def test_measured_sizes(case):
    older, runs = MEASURED[case]
    taken = runs if run(*case)[0] > 0 else older
    assert taken <= 1.08 * min(older, runs)


@pytest.mark.parametrize("zext", [1, 64, 65, 128, 200, 256, 257, 512, 513, 1000])
def test_strips_hold_the_run(zext):
    fn = rules().check_wave_run
    fn.argtypes = [ctypes.c_double] + [ctypes.c_int] * 3 + [ctypes.POINTER(ctypes.c_int)]
    columns = ctypes.c_int()
    for sides in (1, 2):
        for k in range(1, 90):
            zpt = abs(fn(0.05 * k, zext, sides, 32, ctypes.byref(columns)))
            if zpt:
                assert 0.05 * k * (64 * zpt - 1) + 2 + 3 <= columns.value - 2
                assert columns.value - 2 <= 4 * 64 * {8: 3, 4: 2, 2: 1, 1: 1}[zpt] + 3
                assert 16 * sides * columns.value <= 60 * 1024
