"""Products wide and many-rowed enough for the 256 x 128 tile (448 of them and more): remainders of rows, features and depth, one slice
and many, two products in a launch by way of a layer, every epilogue.  Against fp32."""
import pytest
import torch

from tests.test_gpu_layers import _rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("rows,depth,width", [(57601, 72, 264), (57400, 8, 144), (57345, 32, 256), (19201, 200, 776), (28800, 96, 512), (9000, 104, 1792)])
def test_wide_products_match_fp32(rows, depth, width, dtype):
    from dcnv4_amd import ext
    g = torch.Generator(device="cuda").manual_seed(rows)
    rand = lambda *shape: torch.randn(shape, generator=g, device="cuda").to(dtype)
    a, w, b, gamma, res = rand(rows, depth), rand(width, depth) / depth ** 0.5, rand(width), rand(width), rand(rows, width)
    tol = 1e-3 if dtype == torch.float16 else 6e-3        # one rounding to the type
    product = a.float() @ w.float().t()
    got = ext.linear_forward(a, w)
    assert _rel(got, product) < tol and _rel(got[-3:], product[-3:]) < tol and _rel(got[:, -8:], product[:, -8:]) < tol
    want = torch.nn.functional.gelu(product + b.float())
    assert _rel(ext.linear_forward(a, w, b, gelu=True), want) < tol
    assert _rel(ext.linear_forward(a, w, b, gamma, res, gelu=True), want * gamma.float() + res.float()) < tol
