"""filter_wide_kernel at every length it serves (N = 128 .. 16384), with row counts off
the quads, odd widths and the pads, against the oracle's FP64 filter: row-major and
transposed, few rows (a pair at a time) and enough to run two pairs in lockstep, FP32
and FP16 storage.  The bound is the filter's usual one (2e-6 relative RMSE)."""
import numpy as np
import pytest

import fdk_amd as F
import oracle as O

pytestmark = pytest.mark.gpu


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


# N, nu, nrows, views: few rows; then at least 4096 waves of N / 16 threads a row pair
FEW = [(128, 64, 5, 3), (128, 127, 38, 2), (256, 131, 33, 3), (512, 300, 31, 2), (1024, 513, 9, 2),
       (2048, 1024, 7, 3), (4096, 2050, 6, 2), (8192, 4099, 5, 2), (16384, 8200, 3, 1)]
MANY = [(128, 101, 1027, 64), (256, 128, 1030, 32), (512, 257, 1025, 17), (1024, 640, 1031, 8),
        (2048, 1030, 1026, 4), (4096, 2049, 1029, 2), (8192, 4097, 1027, 1)]


def setup(N, nu, nrows, views, seed):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    src = torch.randn((views, nrows, nu), device="cuda", generator=g)
    cos = 0.5 + torch.rand((nrows, nu), device="cuda", generator=g)
    p = F.Parameter(nu=nu, nv=nrows)
    H = p.filter().astype(np.float32)
    assert len(H) == N
    return src, cos, H, torch.as_tensor(H).cuda()


@pytest.mark.parametrize("case", FEW + MANY)
@pytest.mark.parametrize("pad", [F.PAD_MEAN4, F.PAD_ZERO])
def test_matches_oracle(torch_cuda, case, pad):
    import torch
    N, nu, nrows, views = case
    src, cos, H, Hd = setup(*case, seed=N)
    row = torch.empty_like(src)
    tr = torch.full((views, nu, nrows), 7.0, device="cuda")
    F.filter_views(src, row, cos, Hd, pad, False)
    F.filter_views(src, tr, cos, Hd, pad, True)
    torch.cuda.synchronize()
    # rows at both ends of a view's quads, first and last view
    pick = sorted(set(list(range(min(6, nrows))) + list(range(max(0, nrows - 7), nrows))))
    for v in {0, views - 1}:
        x = (src[v, pick] * cos[pick]).cpu().numpy()[None]
        ref = O.filter_rows(x, H.astype(np.float64), pad)[0]
        e1, e2 = rel(row[v, pick].cpu().numpy(), ref), rel(tr[v][:, pick].t().cpu().numpy(), ref)
        print(f"N {N} nu {nu} rows {nrows} views {views} view {v}: {e1:.1e} {e2:.1e}", flush=True)
        assert e1 < 2e-6 and e2 < 2e-6
    assert rel(tr.transpose(1, 2).cpu().numpy(), row.cpu().numpy()) < 2e-6


@pytest.mark.parametrize("case", [(128, 127, 38, 2), (512, 257, 1025, 17), (8192, 4097, 1027, 1)])
def test_16_bit_storage_and_mean3(torch_cuda, case):
    """Per-view min/max and quantization of the same values; no cos table."""
    import torch
    N, nu, nrows, views = case
    src, _, H, Hd = setup(*case, seed=3)
    ref = torch.empty((views, nu, nrows), device="cuda")
    q = torch.empty((views, nu, nrows), dtype=torch.float16, device="cuda")
    F.filter_views(src, ref, None, Hd, F.PAD_MEAN3, True)
    so = F.filter_views(src, q, None, Hd, F.PAD_MEAN3, True, dtype=F.FDK_F16)
    torch.cuda.synchronize()
    lo, hi = ref.amin((1, 2)), ref.amax((1, 2))
    assert np.array_equal(so[:, 1], lo.cpu().numpy())
    assert np.array_equal(so[:, 0], (hi - lo).cpu().numpy())
    want = ((ref - lo[:, None, None]) * (1.0 / (hi - lo))[:, None, None]).half()
    assert float((q.float() - want.float()).abs().max()) <= 2.0 ** -10
    x = src[0, :4].cpu().numpy()[None]
    assert rel(ref[0, :, :4].t().cpu().numpy(), O.filter_rows(x, H.astype(np.float64), F.PAD_MEAN3)[0]) < 2e-6
