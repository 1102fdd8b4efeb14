"""The row filter's blocks of one or two row pairs, taken below two blocks of 256 threads a
CU, against its larger ones: the same rows filtered in one call of many views (large blocks)
and in calls of one view (small ones) give the same bits, at every length that has both
(N = 128 .. 2048), also about the line between them, with odd row counts, and with rows of
NaN and infinities, which reach the other row of their pair and no further."""
import pytest

import fdk_amd as F

pytestmark = pytest.mark.gpu


def filt(src, N, pad, transpose, cos=None):
    import torch
    k = torch.arange(N, device="cuda")
    H = torch.minimum(k, N - k) * (2.0 / N)
    v, nrows, nu = src.shape
    out = torch.full((v, nu, nrows) if transpose else (v, nrows, nu), 7.0, device="cuda")
    F.filter_views(src, out, cos, H, pad, transpose)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("pad", [F.PAD_MEAN4, F.PAD_MEAN3, F.PAD_ZERO])
@pytest.mark.parametrize("N,nu", [(128, 101), (256, 131), (512, 300), (1024, 1000), (2048, 1030)])
def test_small_blocks_equal_large_ones(torch_cuda, N, nu, pad):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(N + pad)
    nrows = 67
    views = 512 * 256 // (N // 16) // 34 + 2  # pairs of two blocks of 256 threads a CU, and over
    src = torch.randn((views, nrows, nu), device="cuda", generator=g)
    src[0, 4] = float("nan")
    src[0, 9, nu // 2] = float("inf")
    src[views - 1, nrows - 1, 0] = float("-inf")  # the last row has no partner
    cos = 0.5 + torch.rand((nrows, nu), device="cuda", generator=g)
    many = filt(src, N, pad, False, cos)
    for v in (0, 1, views - 1):
        for transpose in (False, True):
            one = filt(src[v:v + 1], N, pad, transpose, cos)[0]
            one = one.t() if transpose else one
            assert torch.equal(one.isnan(), many[v].isnan())
            assert torch.equal(torch.nan_to_num(one, 5.0), torch.nan_to_num(many[v], 5.0))
    bad = (~many.isfinite()).any(2).nonzero().tolist()
    assert [v * nrows + r for v, r in bad] == [4, 5, 8, 9, views * nrows - 1]


@pytest.mark.parametrize("N,nu", [(128, 65), (512, 511), (2048, 1500)])
@pytest.mark.parametrize("over", [-1, 0, 1])
def test_about_the_line(torch_cuda, N, nu, over):
    import torch
    pairs = 512 * 256 // (N // 16) + over
    g = torch.Generator(device="cuda")
    g.manual_seed(N)
    src = torch.randn((1, 2 * pairs - 1, nu), device="cuda", generator=g)
    whole = filt(src, N, F.PAD_MEAN4, False)
    part = filt(src[:, :40].contiguous(), N, F.PAD_MEAN4, False)
    assert torch.equal(whole[:, :40], part)
    tail = filt(src[:, -41:].contiguous(), N, F.PAD_MEAN4, False)  # an even row on
    assert torch.equal(whole[:, -41:], tail)
