"""Which form of the row filter a call takes, from the store's offset arithmetic: on the
host, a point that filter_wide_kernel leaves to the resource's range check must fall
outside the view after its 32-bit wrap, for every size the rule gives that form."""
import random

import pytest

from launch_rules import rules

IN_PLACE, WIDE, FAR = 0, 1, 2


def lands_inside(nu, nrows, log_n):
    """Whether some point outside its row has a wrapped offset inside the view."""
    t, view = (1 << log_n) // 16, nu * nrows * 4
    for u in list(range(1 - t, 0)) + list(range(nu, nu + t - 1)):
        first = u * nrows * 4 % 2 ** 32  # of row 0; the other rows follow
        if first < view or first + 4 * nrows > 2 ** 32:
            return True
    return False


def sizes():
    yield from [(512, 1_000_000, 14), (64, 1_030_000, 14), (128, 1 << 21, 14), (4, 1 << 24, 7),
                (5, 65_537, 14), (2048, 2048, 12), (8192, 40_000, 14)]
    rng = random.Random(4)
    for _ in range(300):
        log_n = rng.randrange(7, 15)
        nu = min(1 << log_n, int(2 ** rng.uniform(2, log_n + 0.999)))
        nrows = int(2 ** rng.uniform(0, min(27.0, 30.9 - nu.bit_length())))
        yield nu, max(1, nrows), log_n


@pytest.mark.parametrize("log_n", range(7, 15))
def test_points_outside_the_row_stay_outside_the_view(log_n):
    for nu, nrows, m in sizes():
        if m == log_n and rules().check_filter_form(nu, nrows, 1, m, 1) == WIDE:
            assert not lands_inside(nu, nrows, m), (nu, nrows, m)


def test_ordinary_views_take_the_plain_form():
    for nu, nv, log_n in ((64, 64, 7), (2048, 2048, 12), (4096, 4096, 13), (8192, 8192, 14)):
        assert rules().check_filter_form(nu, nv, 32, log_n, 1) == WIDE
        assert rules().check_filter_form(nu, nv, 32, log_n, 0) == WIDE


@pytest.mark.parametrize("log_n", range(7, 15))
def test_no_view_size_leaves_the_wide_kernel(log_n):
    """Views of 2 GiB and more too: the row-major and 16-bit stores address rows, and the
    transposed FP32 store has its 64-bit form."""
    nu = (1 << log_n) - 3
    for nrows in (300, (1 << 29) // nu, (1 << 29) // nu + 1, 1 << 24):
        assert rules().check_filter_form(nu, nrows, 1, log_n, 0) == WIDE
        big = nu * nrows * 4 >= 2 ** 31
        assert rules().check_filter_form(nu, nrows, 1, log_n, 1) == (FAR if big else WIDE)
    for m in (4, 5, 6):
        assert rules().check_filter_form(20, 30, 1, m, 1) == IN_PLACE
