"""Every form of the RTK-form backprojector's column kernel (two and eight voxels a lane,
with and without paired views) against the general kernel, bit for bit: a z term of 1e-30
in a matrix's row 0 rounds away in every position but selects the general kernel.  Each
case checks that the rule gives it the form it is there for, and that its own matrices
have no z term.  Sizes off the 64-voxel rows and the columns, views of infinities and NaN,
a source inside the volume, samples outside the detector, a matrix that projects nothing."""
import numpy as np
import pytest

import fdk_amd as F
from test_rtk_form_rule import form

pytestmark = pytest.mark.gpu

# volume, detector, pixel, views: form (negative: with pairs)
CASES = {
    "two a lane": ((130, 61, 70), (97, 83), 2.0, 32, 2),
    "two a lane, thin": ((500, 301, 5), (402, 40), 2.0, 8, 2),
    "two a lane, pairs": ((96, 95, 94), (97, 90), 2.2, 32, -2),
    "eight a lane": ((200, 190, 183), (257, 230), 1.6, 2, 8),
    "eight a lane, pairs": ((200, 190, 181), (257, 130), 1.6, 5, -8),
    "eight a lane, pairs, 32 views": ((130, 171, 117), (140, 133), 1.9, 32, -8),
    "detector in the shadow": ((128, 130, 128), (20, 18), 1.5, 32, -8),
}


def steps(p, m):
    x, y = (p.nx - 1) / 2, (p.ny - 1) / 2
    pu = pv = 0.0
    for q in m.astype(np.float64):
        z = 1 / (q[8] * x + q[9] * y + q[11])
        u = (q[0] * x + q[1] * y + q[3]) * z
        pu = max(pu, np.hypot((q[0] - u * q[8]) * z, (q[1] - u * q[9]) * z))
        pv = max(pv, abs(q[6] * z))
    return pu, pv


@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("near", [False, True])
@pytest.mark.parametrize("name", list(CASES))
def test_equals_the_general_kernel(torch_cuda, name, near, special):
    import torch
    (nx, ny, nz), (nu, nv), pixel, views, want = CASES[name]
    p = F.Parameter(nx=nx, ny=ny, nz=nz, nu=nu, nv=nv, du=pixel, dv=pixel, nproj=views, sod=1000.0,
                    sid=1500.0, volume_position_angle_rad=0.3)
    if near:  # the source inside the volume's corners, the centre still magnified by 1.5
        p = p.replace(sod=0.7 * nx, sid=1.05 * nx)
    m = p.proj_matrices().astype(np.float32)
    if special and views > 2:
        m[1] = 0.0
        m[1, 11] = 1.0  # u = v = 0 everywhere
    assert not m[:, 2].any() and not m[:, 10].any()
    assert form(nx, ny, nz, views, nu, nv, *steps(p, m)) == want
    g = torch.Generator(device="cuda")
    g.manual_seed(views + nx)
    proj = torch.randn((views, nv, nu), device="cuda", generator=g)
    if special:
        k = torch.rand(proj.shape, device="cuda", generator=g)
        for part, v in enumerate((float("inf"), float("-inf"), float("nan"), 3e38)):
            proj[(k >= 2e-4 * part) & (k < 2e-4 * (part + 1))] = v
    vin = torch.randn((nz, ny, nx), device="cuda", generator=g)
    out, ref = torch.empty_like(vin), torch.empty_like(vin)
    F.reconstruct_conebeam((nu, nv, views), (nx, ny, nz), m, vin, out, proj)
    m[0, 2] = 1e-30
    F.reconstruct_conebeam((nu, nv, views), (nx, ny, nz), m, vin, ref, proj)
    torch.cuda.synchronize()
    assert torch.equal(out.isnan(), ref.isnan())
    assert torch.equal(torch.nan_to_num(out, 5.0), torch.nan_to_num(ref, 5.0))
    assert not torch.equal(torch.nan_to_num(out, 5.0), vin)


def test_a_matrix_of_nan_off_the_z_columns(torch_cuda):
    """Such a call has no steps to choose a form by, and gives what the general kernel gives."""
    import torch
    n, views = 96, 32
    p = F.Parameter(nx=n, ny=n, nz=n, nu=n, nv=n, du=2.0, dv=2.0, nproj=views)
    m = p.proj_matrices().astype(np.float32)
    m[7, [0, 1, 3, 4, 5, 6, 7, 8, 9, 11]] = np.nan
    proj, vin = torch.randn((views, n, n), device="cuda"), torch.randn((n, n, n), device="cuda")
    out, ref = torch.empty_like(vin), torch.empty_like(vin)
    F.reconstruct_conebeam((n, n, views), (n, n, n), m, vin, out, proj)
    m[0, 2] = 1e-30
    F.reconstruct_conebeam((n, n, views), (n, n, n), m, vin, ref, proj)
    torch.cuda.synchronize()
    assert torch.equal(out, ref) and not torch.equal(out, vin)


def test_captured_pairs_fall_to_two_a_lane(torch_cuda):
    """Nothing is allocated in a capture: the same bits without the pairs."""
    import torch
    n, views = 160, 32
    p = F.Parameter(nx=n, ny=n, nz=n, nu=200, nv=180, du=1.9, dv=1.9, nproj=views)
    m = p.proj_matrices().astype(np.float32)
    assert form(n, n, n, views, 200, 180, *steps(p, m)) == -8
    proj, vin = torch.zeros((views, 180, 200), device="cuda"), torch.randn((n, n, n), device="cuda")
    out = torch.empty_like(vin)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        F.reconstruct_conebeam((200, 180, views), (n, n, n), m, vin, out, proj)
    for _ in range(3):
        proj.copy_(torch.randn_like(proj))
        graph.replay()
        eager = torch.empty_like(out)
        F.reconstruct_conebeam((200, 180, views), (n, n, n), m, vin, eager, proj)
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
