"""The two marches of the forward projector give the same bits: a captured call marches
through the volume itself, the same call outside a capture through the padded copy (the
rule says so), in both edge modes.  Volumes with infinities of one sign, NaN, the largest
floats and negative zeros inside and on every face, sizes off the blocks and a thin volume."""
import pytest

import fdk_amd as F
from test_gpu_fp_runs import takes_the_copy

pytestmark = pytest.mark.gpu

# (nx, ny, nz), (nu, nv), (du, dv), step, first, count
CASES = {
    "odd": ((41, 36, 33), (75, 66), (1.6, 1.0), 0.07, 30, 40),
    "thin": ((40, 47, 2), (80, 65), (1.6, 0.06), 0.03, 20, 60),
    "column": ((3, 2, 50), (64, 130), (0.4, 0.5), 0.002, 0, 60),
    "long steps": ((40, 36, 32), (500, 420), (0.2, 0.2), 3.0, 1, 200),
    "few rows": ((64, 60, 40), (70, 20), (2.0, 2.0), 0.05, 0, 90),
    # a copy past 2 GiB: 64-bit addresses, memory mapped for the call
    "large": ((660, 652, 655), (256, 250), (4.0, 4.2), 0.1, 0, 140),
}


@pytest.mark.parametrize("kind", ["plain", "special"])
@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("mode", [F.FP_CLAMP, F.FP_ZERO])
def test_same_bits(torch_cuda, name, mode, kind):
    import torch
    (nx, ny, nz), (nu, nv), (du, dv), step, first, count = CASES[name]
    p = F.Parameter(nx=nx, ny=ny, nz=nz, nu=nu, nv=nv, du=du, dv=dv, nproj=first + count + 2,
                    volume_position_angle_rad=0.2)
    assert takes_the_copy(p, first, count, step)
    g = torch.Generator(device="cuda")
    g.manual_seed(nx + mode)
    vol = torch.randn((nz, ny, nx), device="cuda", generator=g)
    if kind == "special":
        k = torch.rand(vol.shape, device="cuda", generator=g)
        for part, v in enumerate((float("inf"), float("inf"), float("nan"), 3e38, -0.0, 0.0)):
            vol[(k >= 0.004 * part) & (k < 0.004 * (part + 1))] = v
    direct = torch.empty((count, nv, nu), device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        F.forward_project(p, vol, first, count, direct, step, mode)
    for _ in range(2):
        direct.zero_()
        graph.replay()
        out = torch.empty_like(direct)
        F.forward_project(p, vol, first, count, out, step, mode)
        torch.cuda.synchronize()
        print(name, mode, kind, int((out != direct).sum()), flush=True)
        assert torch.equal(out.isnan(), direct.isnan())
        assert torch.equal(torch.nan_to_num(out, 5.0), torch.nan_to_num(direct, 5.0))
    assert float((direct != 0).float().mean()) > 0.02
