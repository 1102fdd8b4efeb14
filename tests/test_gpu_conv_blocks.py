"""The forward convolution's tiles a block (one, or two where the launch fills whole rounds
of resident blocks): a batch whose tile count falls on either side of the rule gives, image
by image, the bits of the images alone."""
import numpy as np
import pytest

import fdk_amd  # noqa: F401
from fdk_amd import unet as U

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cin", [32, 96])
@pytest.mark.parametrize("images", [24, 25, 31, 32, 33, 57])
def test_batches_equal_their_images(torch_cuda, cin, images):
    import torch
    cv = U.Conv3(cin, 32, 1, np.random.default_rng(1), "cuda")
    cv.refresh()
    g = torch.Generator(device="cuda")
    g.manual_seed(images)
    x = torch.randn((images, 4, 64, 64, cin), device="cuda", generator=g).bfloat16().view(torch.int16)
    many = cv.forward(x, (images, 4, 64, 64))  # 32 tiles an image
    for k in (0, images // 2, images - 1):
        one = cv.forward(x[k:k + 1].contiguous(), (1, 4, 64, 64))
        torch.cuda.synchronize()
        assert torch.equal(many[k], one.view(many[k].shape))
    assert int((many != 0).sum()) > many.numel() // 4
