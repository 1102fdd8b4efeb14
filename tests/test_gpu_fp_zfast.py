"""The z-fastest forward projector (taken where a scan's samples outweigh the padded
copy it reads) in both edge modes: odd and thin volumes, detector sizes off the block,
steps far below and above a voxel, a view range inside the scan.

A captured call allocates nothing and marches the volume as it is (fp_kernel), with the
same positions: both sum the same samples, so every pixel agrees to the rounding of a
blend (a few 1e-7 of the largest sum; the bound is 1e-5).  The oracle marches in FP64,
where a step that is no binary fraction drifts from the FP32 additions by up to 3e-5 mm
a step, so it is compared at a step of 1/16 mm."""
import numpy as np
import pytest

import fdk_amd as F
import oracle as O

pytestmark = pytest.mark.gpu

# (nx, ny, nz), (nu, nv), du, step, first, count
CASES = {
    "odd": ((41, 36, 33), (75, 66), 1.6, 0.07, 3, 9),
    "thin": ((40, 47, 2), (80, 65), 1.6, 0.03, 0, 12),
    "column": ((3, 2, 50), (64, 130), 0.4, 0.002, 0, 12),
    "long steps": ((40, 36, 32), (500, 420), 0.2, 11.0, 1, 60),
}


def scan(case):
    (nx, ny, nz), (nu, nv), du, step, first, count = CASES[case]
    p = F.Parameter(nx=nx, ny=ny, nz=nz, nu=nu, nv=nv, du=du, dv=du, nproj=first + count + 2,
                    volume_position_angle_rad=0.2)
    return p, step, first, count


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("mode", [F.FP_CLAMP, F.FP_ZERO])
def test_equals_the_march_through_the_volume_itself(torch_cuda, name, mode):
    import torch
    p, step, first, count = scan(name)
    vol = torch.zeros((p.nz, p.ny, p.nx), device="cuda")
    direct = torch.empty((count, p.nv, p.nu), device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        F.forward_project(p, vol, first, count, direct, step, mode)
    for seed in range(3):
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        vol.copy_(torch.rand(vol.shape, device="cuda", generator=g))
        direct.zero_()
        graph.replay()
        out = torch.empty_like(direct)
        F.forward_project(p, vol, first, count, out, step, mode)
        torch.cuda.synchronize()
        far = float((out - direct).abs().max()) / float(direct.abs().max())
        print(f"{name} mode {mode} seed {seed}: {far:.1e}", flush=True)
        assert far <= 1e-5


@pytest.mark.parametrize("mode", [F.FP_CLAMP, F.FP_ZERO])
def test_matches_oracle(torch_cuda, mode):
    import torch
    p, _, first, count = scan("odd")
    step = 1.0 / 16
    vol = np.random.default_rng(5).random((p.nz, p.ny, p.nx)).astype(np.float32)
    out = torch.empty((count, p.nv, p.nu), device="cuda")
    F.forward_project(p, torch.as_tensor(vol).cuda(), first, count, out, step, mode)
    torch.cuda.synchronize()
    g = O.Geom(**{k: getattr(p, k) for k in O.Geom.__dataclass_fields__})
    views = [0, count // 3, count - 1]
    ref = np.stack([O.fp(g, vol, first + s, step, mode) for s in views])
    got = out[views].cpu().numpy()
    frac = float((np.abs(got - ref) <= 1e-4 * np.abs(ref).max()).mean())
    print(f"mode {mode}: {frac:.4f} of pixels within 1e-4", flush=True)
    assert frac > 0.995
