"""16-bit views that no 4-byte load fits -- odd rows, odd view strides, odd
addresses -- on volumes large enough for the re-pitched copy and on one that is not
(the gathers straight from memory), against the FP32 path on the same values, slab
by slab: a mirror pair of rows of a multiple of four samples takes the mirrored
position there, which these views never did.

Both sides round positions in FP32 (about 1e-5 px here) on views whose samples
are independent, the bound of the other wave-kernel tests: 2e-5 relative RMSE."""
import numpy as np
import pytest

import fdk_amd as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [F.FDK_F16, F.FDK_BF16])
@pytest.mark.parametrize("nv,shift,gap,pair", [(97, 0, 0, True), (99, 0, 1, False), (96, 1, 0, True),
                                               (98, 0, 1, False), (101, 1, 3, True)])
@pytest.mark.parametrize("n", [150, 24])
def test_rows_off_four_bytes(torch_cuda, dtype, nv, shift, gap, pair, n):
    torch = torch_cuda
    nu, views, nz = 110, 32, 120
    p = F.Parameter(nx=n, ny=n - 9, nz=nz, dx=1.0, dy=1.0, dz=1.0, nu=nu, nv=nv, du=1.6, dv=1.4, nproj=views,
                    filter_type=5, volume_position_angle_rad=0.15)
    t = torch.float16 if dtype == F.FDK_F16 else torch.bfloat16
    g = torch.Generator("cuda").manual_seed(nv + n)
    q = torch.rand((views, nu, nv), generator=g, device="cuda").to(t)
    stride = nu * nv + gap
    buf = torch.full((views * stride + shift,), float("nan"), dtype=t, device="cuda")
    odd = buf[shift:].view(views, stride)
    odd[:, :nu * nv] = q.view(views, -1)
    so = np.stack([np.linspace(0.5, 2.0, views), np.linspace(-0.2, 0.3, views)], 1).astype(np.float32)
    sc = torch.as_tensor(so).cuda()
    full = q.float() * sc[:, 0, None, None] + sc[:, 1, None, None]
    mats = p.proj_matrices().astype(np.float32)
    top = (0, 0, 0, p.nx, p.ny, nz // 2)
    bottom = (0, 0, nz // 2, p.nx, p.ny, nz // 2) if pair else (0,) * 6

    def run(data, dt, vs, scale, top, bottom=(0,) * 6):
        bp = F.BackProjectionFDK(nv, nu, views, p.nx, p.ny, nz, top, bottom)
        bp.set_stream(torch.cuda.current_stream().cuda_stream)
        bp.bp_device(data, nv, nu, mats, views, dtype=dt, view_stride=vs, scale_offset=scale)
        bp.sync()
        v = bp.GetVolumeData()
        bp.close()
        return v

    ref = np.concatenate([run(full.contiguous(), F.FDK_F32, nu * nv, None, b) for b in (top, bottom) if b[5]])
    got = run(buf[shift:], dtype, stride, so, top, bottom)
    err = float(np.linalg.norm(got - ref) / np.linalg.norm(ref))
    print(f"{n} {nv} {shift} {gap} {pair} {dtype}: {err:.2e}", flush=True)
    assert err < 2e-5
