"""The wave-strip backprojector's run lengths and edges, against the oracle's
strict-bilinear backprojection: single-slab runs of every length (64 .. 512
voxels, cut inside a run), mirror pairs of every length, a pair whose matrices
are not mirror-symmetric, grids small enough to split the views over a block's
waves, edge tiles, and detector rows that are no multiple of four samples, with
columns projecting onto the view's first and last rows.

The bound is that of the other wave-kernel tests: positions are FP32 (about 1e-5
px of rounding on these detectors) and the projections' edges are a pixel wide,
2e-5 relative RMSE."""
import numpy as np
import pytest

import fdk_amd as F
import oracle as O

pytestmark = pytest.mark.gpu


def views_of(p, seed=11):
    import torch
    ext = max(p.nx, p.ny, 40) * p.dx
    ell = F.random_ellipsoids(8, seed=seed, radius_mm=0.4 * ext,
                              half_height_mm=0.45 * max(p.nz, 20) * p.dz,
                              axes_mm=(4 * p.dx, 0.3 * ext))
    raw = torch.empty((p.nproj, p.nv, p.nu), device="cuda")
    F.phantom_project(ell, p, 0, p.nproj, raw)
    return raw.cpu().numpy()


def reconstruct(p, proj, mats, top, bottom, dtype=F.FDK_F32):
    import torch
    v = torch.as_tensor(np.ascontiguousarray(proj.transpose(0, 2, 1))).cuda()
    so = None
    if dtype != F.FDK_F32:
        lo, hi = v.amin((1, 2)), v.amax((1, 2))
        q = (v - lo[:, None, None]) / (hi - lo)[:, None, None]
        q = q.half() if dtype == F.FDK_F16 else q.bfloat16()
        so = torch.stack([hi - lo, lo], 1).cpu().numpy()
        proj = (q.float() * (hi - lo)[:, None, None] + lo[:, None, None]).transpose(1, 2)
        proj, v = proj.contiguous().cpu().numpy(), q.contiguous()
    bp = F.BackProjectionFDK(p.nv, p.nu, 32, p.nx, p.ny, p.nz, top, bottom)
    bp.set_stream(torch.cuda.current_stream().cuda_stream)
    for b in range(0, p.nproj, 32):
        n = min(32, p.nproj - b)
        bp.bp_device(v, p.nv, p.nu, mats[b:b + n], n, dtype=dtype, offset_views=b,
                     scale_offset=None if so is None else so[b:b + n])
    bp.sync()
    vol = bp.GetVolumeData()
    bp.close()
    return vol, proj


def check(p, top, bottom, dtype=F.FDK_F32, shift=0.0):
    proj = views_of(p)
    m = p.proj_matrices()
    m[:, 4:8] += shift * m[:, 8:12]  # v + shift pixels
    mats = m.astype(np.float32)
    vol, proj = reconstruct(p, proj, mats, top, bottom, dtype)
    g = O.Geom(**{k: getattr(p, k) for k in O.Geom.__dataclass_fields__})
    ref = np.concatenate([O.bp(g, proj, mats.astype(np.float64), O.BP_GPU_STRICT, z0=b[2], nzs=b[5])
                          for b in (top, bottom) if b[5]])
    err = float(np.linalg.norm(vol - ref) / np.linalg.norm(ref))
    print(f"{p.nx}x{p.ny}x{p.nz} {p.nu}x{p.nv} dtype {dtype}: {err:.2e}", flush=True)
    assert err < 2e-5


def scan(nx, ny, nz, nu, nv, views=34, **kw):
    return F.Parameter(nx=nx, ny=ny, nz=nz, dx=1.0, dy=1.0, dz=1.0, nu=nu, nv=nv,
                       du=1.7 * max(nx, ny, 40) / nu, dv=1.5, nproj=views, filter_type=5,
                       volume_position_angle_rad=0.15, **kw)


@pytest.mark.parametrize("depth", [1, 63, 65, 129, 300, 513])
@pytest.mark.parametrize("pair", [False, True])
def test_run_lengths(torch_cuda, depth, pair):
    nz = 2 * depth + 10
    p = scan(70, 67, nz, 96, max(64, (nz // 4) * 4))
    top = (0, 0, 5, p.nx, p.ny, depth)
    check(p, top, (0, 0, 5 + depth, p.nx, p.ny, depth) if pair else (0,) * 6)


@pytest.mark.parametrize("shape", [(1, 1), (3, 5), (33, 2), (20, 40), (66, 64)])
def test_small_and_edge_grids(torch_cuda, shape):
    """Split views (few columns), single columns, cut tiles; 7 views are not split."""
    for views in (7, 9, 32):
        p = scan(shape[0], shape[1], 70, 80, 96, views=views)
        check(p, (0, 0, 0, p.nx, p.ny, 35), (0, 0, 35, p.nx, p.ny, 35))
        check(p, (0, 0, 3, p.nx, p.ny, 60), (0,) * 6)


@pytest.mark.parametrize("nv", [61, 62, 63, 97])
@pytest.mark.parametrize("dtype", [F.FDK_F32, F.FDK_F16, F.FDK_BF16])
def test_rows_not_a_multiple_of_four(torch_cuda, nv, dtype):
    """Narrow detector (nu = 40): columns project onto its first and last rows."""
    p = scan(64, 60, 80, 40, nv).replace(du=1.5)
    check(p, (0, 0, 0, p.nx, p.ny, 40), (0, 0, 40, p.nx, p.ny, 40), dtype)
    check(p, (0, 0, 10, p.nx, p.ny, 70), (0,) * 6, dtype)


@pytest.mark.parametrize("dtype", [F.FDK_F32, F.FDK_F16])
def test_pair_without_mirror_symmetry(torch_cuda, dtype):
    p = scan(48, 50, 120, 64, 100)
    check(p, (0, 0, 0, p.nx, p.ny, 60), (0, 0, 60, p.nx, p.ny, 60), dtype, shift=2.5)
