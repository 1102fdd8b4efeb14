"""The volume's way out of the handle, [x][y][z] to [z][y][x]: every voxel of the
handle's own array at its place, for whole and cut tiles of the 16-byte form and
for sizes and destinations that it does not take."""
import numpy as np
import pytest

import fdk_amd as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz,shift", [(64, 3, 64, 0), (128, 2, 192, 0), (68, 5, 132, 0), (4, 7, 4, 0),
                                            (60, 3, 124, 0), (68, 5, 130, 0), (66, 5, 132, 0), (68, 5, 132, 1)])
def test_volume_out(torch_cuda, nx, ny, nz, shift):
    torch = torch_cuda
    bp = F.BackProjectionFDK(8, 8, 1, nx, ny, nz, (0, 0, 0, nx, ny, nz), (0, 0, 0, 0, 0, 0))
    vol = bp.volume_tensor()
    vol.copy_(torch.arange(vol.numel(), device="cuda", dtype=torch.float32).view(vol.shape))
    torch.cuda.synchronize()
    buf = torch.full((nz * ny * nx + shift,), -1.0, device="cuda")
    out = buf[shift:].view(nz, ny, nx)
    bp.get_volume_device(out)
    ref = vol.permute(2, 1, 0)
    assert torch.equal(out, ref)
    assert np.array_equal(bp.GetVolumeData().reshape(nz, ny, nx), ref.cpu().numpy())
    bp.close()
