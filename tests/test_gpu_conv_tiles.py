"""3x3x3 convolution layers: the work split of the forward and weight-gradient
kernels and the fused activation adjoint and bias gradient, against the FP64
restatement."""
import numpy as np
import pytest

import fdk_amd.unet as U
from oracle import nn_ref as R

pytestmark = pytest.mark.gpu


def bf(torch, a):
    return torch.as_tensor(R.to_bf16_bits(a).view(np.int16)).cuda()


def from_bf(t):
    return R.from_bf16_bits(t.cpu().numpy().view(np.uint16))


def rel(a, b):
    return float(np.linalg.norm(np.ravel(a - b)) / max(np.linalg.norm(np.ravel(b)), 1e-300))


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("c,nvox,shift", [(16, 4099, 0), (32, 1, 0), (32, 70001, 0), (64, 3 * 4099, 0),
                                          (128, 5003, 0), (128, 5003, 1)])
def test_activation_and_bias(torch_cuda, c, nvox, shift, mode):
    """dz bit for bit (dy where y > 0, else 0 or 0.01 dy rounded to BF16) and its
    per-channel sums added to db: the one-pass form at 32, 64 and 128 channels,
    the two kernels at 16 channels and for a tensor off 16-byte alignment."""
    torch = torch_cuda
    rng = np.random.default_rng(c + nvox + mode)
    dy = R.bf16_round(rng.standard_normal((nvox, c)))
    y = R.bf16_round(rng.standard_normal((nvox, c)))
    y[::7] = 0.0
    ref = np.where(y > 0, dy, 0.0 if mode == 1 else R.bf16_round(np.float32(0.01) * dy.astype(np.float32)))
    buf = torch.empty(nvox * c + shift, dtype=torch.int16, device="cuda")
    g = buf[shift:].view(nvox, c)
    g.copy_(bf(torch, dy))
    dz = torch.empty((nvox, c), dtype=torch.int16, device="cuda")
    db = torch.ones(c, device="cuda")
    U.act_bias_bwd(g, bf(torch, y), dz, db, nvox, c, mode)
    assert np.array_equal(from_bf(dz), ref)
    # FP32 sums: at most nvox roundings of 2^-24 of the sum of magnitudes, in practice their root
    bound = (1.0 + np.abs(ref).sum(0)) * 2.0 ** -24 * (8.0 + nvox ** 0.5)
    assert (np.abs(db.cpu().numpy() - (1.0 + ref.sum(0))) <= bound).all()


@pytest.mark.parametrize("cin,cout,n", [(32, 32, 3), (96, 32, 70), (288, 160, 13), (1216, 256, 3)])
def test_weight_gradient_block_counts(torch_cuda, cin, cout, n):
    """Weight gradients over 1, 3, 45 and 304 channel chunks, with 3, 30, 3 and 1
    blocks a chunk: tiles that the blocks do not share evenly, one block for all."""
    torch = torch_cuda
    shape = (n, 2, 4, 32)
    rng = np.random.default_rng(cin)
    x = R.bf16_round(rng.standard_normal(shape + (cin,)))
    dy = R.bf16_round(rng.standard_normal(shape + (cout,)))
    dw = torch.zeros((27, cout, cin), device="cuda")
    U.conv3d_wgrad(bf(torch, x), bf(torch, dy), dw, shape, cin, cout)
    assert rel(dw.cpu().numpy(), R.conv3d_dw(x, dy)) < 1e-5


@pytest.mark.parametrize("cout", [64, 96, 128, 224])
def test_forward_passes(torch_cuda, cout):
    """1, 1, 2 and 3 passes of 64 output channels in one launch, and the 32 that
    96 and 224 leave."""
    torch = torch_cuda
    rng = np.random.default_rng(cout)
    shape = (1, 4, 8, 64)
    x = R.bf16_round(rng.standard_normal(shape + (32,)))
    w = R.bf16_round(rng.standard_normal((27, cout, 32)) / np.sqrt(27 * 32))
    b = rng.standard_normal(cout).astype(np.float32)
    y = torch.empty(shape + (cout,), dtype=torch.float32, device="cuda")
    U.conv3d(bf(torch, x), bf(torch, w), torch.as_tensor(b).cuda(), y, shape, 32, cout, relu=False, out_f32=True)
    assert rel(y.cpu().numpy(), R.conv3d(x, w, b)) < 1e-5


@pytest.mark.parametrize("n", [8191, 8193])
def test_forward_tiles_per_block(torch_cuda, n):
    """One tile a block below 8192 tiles and two from there on (an odd count):
    every sample equals, bit for bit, the same sample computed by itself."""
    torch = torch_cuda
    rng = np.random.default_rng(n)
    s = bf(torch, R.bf16_round(rng.standard_normal((3, 4, 4, 32, 32))))
    w = bf(torch, R.bf16_round(rng.standard_normal((27, 32, 32)) / np.sqrt(27 * 32)))
    one = torch.empty((3, 4, 4, 32, 32), dtype=torch.int16, device="cuda")
    U.conv3d(s, w, None, one, (3, 4, 4, 32), 32, 32, relu=True)
    k = torch.arange(n, device="cuda") % 3
    y = torch.empty((n, 4, 4, 32, 32), dtype=torch.int16, device="cuda")
    U.conv3d(s[k].contiguous(), w, None, y, (n, 4, 4, 32), 32, 32, relu=True)
    assert torch.equal(y, one[k])
