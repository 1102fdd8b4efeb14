"""Which march of the forward projector a call takes, against the times measured both
ways (microseconds: fp_kernel, fp_zfast_kernel with its copy): nowhere the slower march,
by more than the spread of a measurement, where fp_kernel is the faster, and the copy
wherever it wins by two and a quarter.  Volumes n x n x nz of 256 mm, detectors n x nv, `views`
views round the scan or (arc) of a 720-view scan from 0.1 rad on."""
import ctypes
import math

import pytest

from launch_rules import rules

# n, nz, nv, views, arc, step in voxels: fp_kernel, fp_zfast_kernel
MEASURED = {
    (64, 64, 1, 60, True, 0.5): (23, 47), (64, 64, 16, 60, True, 0.5): (27, 43),
    (64, 64, 200, 24, False, 0.5): (162, 59), (128, 128, 64, 360, False, 0.5): (3184, 640),
    (128, 128, 80, 24, True, 0.5): (121, 115), (128, 128, 128, 8, False, 0.5): (227, 73),
    (128, 128, 200, 1, True, 0.5): (40, 71), (256, 256, 1, 360, True, 0.5): (268, 2400),
    (256, 256, 8, 60, False, 0.5): (521, 548), (256, 256, 8, 360, False, 0.5): (1902, 2400),
    (256, 256, 16, 60, False, 0.5): (686, 524), (256, 256, 64, 24, False, 0.5): (1216, 260),
    (256, 256, 64, 360, False, 0.5): (14763, 2601), (256, 256, 80, 24, False, 0.5): (1382, 415),
    (256, 256, 200, 2, True, 0.5): (124, 152), (256, 256, 200, 24, False, 0.5): (3734, 716),
    (400, 400, 80, 1, True, 0.5): (154, 472), (400, 400, 200, 4, False, 0.5): (1239, 692),
    (256, 1, 16, 60, False, 0.5): (19, 24), (256, 1, 64, 360, False, 0.5): (36, 49),
    (512, 1, 1, 360, False, 0.5): (975, 9182), (512, 1, 64, 360, False, 0.5): (70, 96),
    (512, 1, 100, 60, False, 0.5): (21, 46), (512, 16, 1, 360, False, 0.5): (1031, 9162),
    (512, 16, 64, 360, False, 0.5): (33930, 9167), (512, 16, 100, 60, False, 0.5): (5786, 3182),
    # whole steps, few views
    (84, 90, 90, 4, False, 1.0): (19.4, 29.6), (98, 95, 103, 3, False, 1.0): (34.0, 36.2),
    (160, 167, 169, 3, False, 1.0): (140, 61), (190, 186, 188, 3, False, 1.0): (291, 76),
    # waited for, call by call
    (300, 300, 300, 1, False, 1.0): (102, 204), (300, 300, 300, 8, False, 1.0): (1422, 371),
    (400, 400, 400, 1, False, 1.0): (177, 429), (400, 400, 400, 8, False, 1.0): (2940, 971),
    (512, 512, 512, 1, False, 1.0): (333, 1144), (512, 512, 512, 8, False, 1.0): (7250, 26813),
    (700, 700, 700, 8, False, 1.0): (18914, 68673), (1024, 1024, 1024, 8, False, 1.0): (126334, 483481),
}


def pays(n, nz, nv, views, arc, step):
    fn = rules().check_zfast_pays
    d, i = ctypes.c_double, ctypes.c_int
    fn.argtypes = [i, i, d, d, i, i, d, d, i, d, d]
    vox = 256.0 / n
    sines = [abs(math.sin(0.1 + 2 * math.pi * k / (720 if arc else views))) for k in range(views)]
    return bool(fn(n, nv, (nv - 1) / 2, 1.62 * vox * 0.6, n, nz, vox, step * vox, views, sum(sines), max(sines)))


@pytest.mark.parametrize("case", list(MEASURED))
def test_measured_sizes(case):
    direct, zfast = MEASURED[case]
    if pays(*case):
        assert zfast <= 1.04 * direct
    else:
        assert direct <= 2.25 * zfast


@pytest.mark.parametrize("n", [64, 256, 512])
@pytest.mark.parametrize("nv", [1, 4, 8])
@pytest.mark.parametrize("views", [1, 60, 1000])
def test_few_detector_rows_march_through_the_volume(n, nv, views):
    assert not pays(n, n, nv, views, False, 0.5)


@pytest.mark.parametrize("views", [360, 1000])
def test_whole_scans_of_large_volumes_take_the_copy(views):
    assert pays(512, 512, 512, views, False, 1.0) and pays(1024, 1024, 1024, views, False, 1.0)
