"""Views much shorter than the filter's length N and so tall that the 32-bit offsets of
points outside their rows would wrap into the view: the transposed store checks them.
The row-major form stores through one resource a row and runs the same transform, so
the two outputs are equal to the bit."""
import pytest

import fdk_amd as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nu,nrows", [(512, 1_000_000), (64, 1_030_001)])
def test_transposed_equals_row_major(torch_cuda, nu, nrows):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(nu)
    src = torch.randn((1, nrows, nu), device="cuda", generator=g)
    k = torch.arange(16384, device="cuda")
    H = torch.minimum(k, 16384 - k) / 8192.0
    row = torch.empty_like(src)
    tr = torch.full((1, nu, nrows), 7.0, device="cuda")
    print(f"nu {nu} rows {nrows}", flush=True)
    F.filter_views(src, row, None, H, F.PAD_MEAN4, False)
    F.filter_views(src, tr, None, H, F.PAD_MEAN4, True)
    torch.cuda.synchronize()
    assert torch.equal(tr[0].t(), row[0])


@pytest.mark.parametrize("nu,parts", [(1000, 9), (300, 31)])
def test_views_of_2_gib_equal_their_parts(torch_cuda, nu, parts):
    """A view of 2 GiB and more against the same rows as several smaller views."""
    import torch
    nrows = ((1 << 29) // nu // parts + 3) // 2 * 2 * parts  # an even number of rows a part
    assert nu * nrows * 4 >= 1 << 31
    g = torch.Generator(device="cuda")
    g.manual_seed(nu)
    src = torch.randn((nrows, nu), device="cuda", generator=g)
    N = 1 << nu.bit_length()
    k = torch.arange(N, device="cuda")
    H = torch.minimum(k, N - k) * (2.0 / N)
    print(f"nu {nu} rows {nrows}", flush=True)
    ref = torch.empty((parts, nrows // parts, nu), device="cuda")
    F.filter_views(src.view(ref.shape), ref, None, H, F.PAD_MEAN3, False)
    ref = ref.view(nrows, nu)
    out = torch.full((1, nrows, nu), 7.0, device="cuda")
    F.filter_views(src[None], out, None, H, F.PAD_MEAN3, False)
    torch.cuda.synchronize()
    assert torch.equal(out[0], ref)
    out = out.view(1, nu, nrows).fill_(7.0)
    F.filter_views(src[None], out, None, H, F.PAD_MEAN3, True)
    torch.cuda.synchronize()
    assert torch.equal(out[0].t(), ref)
