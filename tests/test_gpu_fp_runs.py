"""A forward projection of more blocks than a launch takes (2^22) is cut into runs of
views: the views about the cuts equal the same views projected in calls of their own,
which are single launches of the same march."""
import ctypes
import math

import pytest

import fdk_amd as F
from launch_rules import rules

pytestmark = pytest.mark.gpu


def takes_the_copy(p, first, count, step):
    fn = rules().check_zfast_pays
    d, i = ctypes.c_double, ctypes.c_int
    fn.argtypes = [i, i, d, d, i, i, d, d, i, d, d]
    sines = [abs(math.sin(p.view_angle(first + k))) for k in range(count)]
    return bool(fn(p.nu, p.nv, (p.nv - 1) / 2, p.dv, p.nx, p.nz, p.dx, step, count, sum(sines), max(sines)))


def test_views_about_the_cut(torch_cuda):
    import torch
    p = F.Parameter(nx=24, ny=24, nz=24, nu=1020, nv=250, du=0.05, dv=0.2, nproj=16000)
    most = (1 << 22) // (4 * 255)  # views of a launch
    count, step = most + 40, 0.05
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    vol = torch.rand((24, 24, 24), device="cuda", generator=g)
    out = torch.empty((count, p.nv, p.nu), device="cuda")
    assert takes_the_copy(p, 3, count, step)
    F.forward_project(p, vol, 3, count, out, step)
    for v in (most - 30, most, count - 30):
        assert takes_the_copy(p, 3 + v, 30, step)
        ref = torch.empty((30, p.nv, p.nu), device="cuda")
        F.forward_project(p, vol, 3 + v, 30, ref, step)
        torch.cuda.synchronize()
        assert torch.equal(out[v:v + 30], ref)
        assert float(ref.abs().max()) > 1
