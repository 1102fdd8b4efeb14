"""The ratio loop's quotient kernels against the element-wise form, bit for bit:
zero, infinite and NaN operands, odd sizes, and the arrays that keep that form."""
import pytest

import fdk_amd.iterative as it

pytestmark = pytest.mark.gpu


def operands(torch, shape, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    a, b = (torch.randn(shape, generator=g, device="cuda") for _ in range(2))
    inf, nan = float("inf"), float("nan")
    special = torch.tensor([0.0, -0.0, inf, -inf, nan, 1e-40, 3e38], device="cuda")
    k = torch.randint(0, 21, shape, generator=g, device="cuda")
    for t, q in ((a, k % 7), (b, k // 3)):
        pick = torch.rand(shape, generator=g, device="cuda") < 0.3
        t[pick] = special[q[pick]]
    return a, b


def same(torch, x, y):
    return x.dtype == y.dtype and torch.equal(torch.nan_to_num(x, 7.0), torch.nan_to_num(y, 7.0)) \
        and torch.equal(x.isnan(), y.isnan())


@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 17, 31), (1030, 5, 7), (2, 300, 257)])
def test_quotients(torch_cuda, shape):
    torch = torch_cuda
    a, b = operands(torch, shape, sum(shape))
    m = (torch.arange(shape[1] * shape[2], device="cuda") % 3 > 0).float().view(shape[1:])
    assert same(torch, it._masked_ratio(a, b, m), it._safe_div(a, b) * m)
    x = torch.randn(shape, device="cuda")
    ref = x * it._safe_div(a, b)
    assert it._scale_by_ratio(x, a, b) is x and same(torch, x, ref)


def test_other_arrays(torch_cuda):
    torch = torch_cuda
    a, b = operands(torch, (4, 6, 10), 5)
    m = torch.ones((6, 10), device="cuda")
    t = a.transpose(1, 2).contiguous().transpose(1, 2)
    assert same(torch, it._masked_ratio(t, b, m), it._masked_ratio(a, b, m))
    assert same(torch, it._masked_ratio(a.double(), b, m), it._safe_div(a.double(), b) * m)
    x = torch.randn((10, 6, 4), device="cuda").permute(2, 1, 0)
    ref = x * it._safe_div(a, b)
    assert same(torch, it._scale_by_ratio(x, a, b), ref)
