"""Backprojection passes of one to four views, which take the wave-strip kernel, the
block-strip kernel or the gather kernel by storage, row length and size: pairs with and
without 4-sample rows, single slabs, FP32 and FP16, grids on both sides of the rule's
line for single views.  Oracle and bound are those of the wave-strip tests."""
import pytest

import fdk_amd as F
from test_gpu_wave_runs import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("views", [1, 2, 3, 4])
@pytest.mark.parametrize("nv", [56, 57, 58])
@pytest.mark.parametrize("dtype", [F.FDK_F32, F.FDK_F16])
@pytest.mark.parametrize("pair", [True, False])
def test_few_views(torch_cuda, views, nv, dtype, pair):
    p = F.Parameter(nx=45, ny=42, nz=40, nu=61, nv=nv, du=1.3, dv=1.3, nproj=views)
    top = (0, 0, 0, 45, 42, 20 if pair else 40)
    check(p, top, (0, 0, 20, 45, 42, 20) if pair else (0, 0, 0, 0, 0, 0), dtype)


@pytest.mark.parametrize("nv", [32, 33])
@pytest.mark.parametrize("pair", [True, False])
def test_one_view_on_many_columns(torch_cuda, nv, pair):
    p = F.Parameter(nx=290, ny=284, nz=12, nu=330, nv=nv, du=1.5, dv=1.5, nproj=1)
    top = (0, 0, 0, 290, 284, 6 if pair else 12)
    check(p, top, (0, 0, 6, 290, 284, 6) if pair else (0, 0, 0, 0, 0, 0))
