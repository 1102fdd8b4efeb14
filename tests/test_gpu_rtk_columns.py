"""The RTK-form backprojector's column kernel against its general kernel: a z term of
1e-30 in a matrix's row 0 rounds away in every position but selects the general kernel,
so the two volumes are equal to the bit (the sums run over the same views in the same
order).  Sizes off the 64-voxel rows, the 2- and 8-voxel columns and the 256-sample pair
rows, few and many views, a detector smaller than the volume's shadow, a source inside
the volume, and a matrix of NaN."""
import numpy as np
import pytest

import fdk_amd as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vol,det,views", [
    ((130, 61, 70), (97, 83), 32),     # two voxels a lane, no pairs
    ((200, 190, 181), (257, 130), 5),  # eight voxels a lane, pairs, nz % 8 == 5
    ((65, 200, 100), (64, 300), 17),
    ((128, 128, 128), (20, 18), 32),   # most voxels outside the detector
])
@pytest.mark.parametrize("near", [False, True])
def test_equals_the_general_kernel(torch_cuda, vol, det, views, near):
    import torch
    nx, ny, nz = vol
    p = F.Parameter(nx=nx, ny=ny, nz=nz, nu=det[0], nv=det[1], du=1.5, dv=1.5, nproj=views,
                    sod=40.0 if near else 1000.0, sid=60.0 if near else 1500.0,
                    volume_position_angle_rad=0.3)
    m = p.proj_matrices().astype(np.float32)
    if views > 16:
        m[7] = np.nan
    g = torch.Generator(device="cuda")
    g.manual_seed(2)
    proj = torch.randn((views, det[1], det[0]), device="cuda", generator=g)
    vin = torch.randn((nz, ny, nx), device="cuda", generator=g)
    out, ref = torch.empty_like(vin), torch.empty_like(vin)
    F.reconstruct_conebeam((det[0], det[1], views), vol, m, vin, out, proj)
    m[0, 2] = 1e-30
    F.reconstruct_conebeam((det[0], det[1], views), vol, m, vin, ref, proj)
    torch.cuda.synchronize()
    assert torch.equal(out, ref)
    assert not torch.equal(out, vin)


def test_captured_call(torch_cuda):
    """Nothing is allocated in a capture: the views are gathered as they are."""
    import torch
    p = F.Parameter(nx=160, ny=150, nz=140, nu=200, nv=180, nproj=32)
    m = p.proj_matrices().astype(np.float32)
    proj = torch.zeros((32, 180, 200), device="cuda")
    vin = torch.zeros((140, 150, 160), device="cuda")
    out = torch.empty_like(vin)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        F.reconstruct_conebeam((200, 180, 32), (160, 150, 140), m, vin, out, proj)
    for k in range(3):
        proj.copy_(torch.randn_like(proj))
        graph.replay()
        eager = torch.empty_like(out)
        F.reconstruct_conebeam((200, 180, 32), (160, 150, 140), m, vin, eager, proj)
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
