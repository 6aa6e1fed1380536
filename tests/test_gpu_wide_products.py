"""Products wide and many-rowed enough for the 256 x 128 tile (448 of them and more): remainders of rows, features and depth, one slice
and many, and the inference epilogues, against fp32; two products in a launch and what training adds to the epilogue by way of a
layer, against its composition."""
import pytest
import torch

from tests.test_gpu_layers import _composed, _rel

pytestmark = pytest.mark.gpu


def _tile(rows, depth, *widths, result32=0):
    from dcnv4_amd import ext
    return ext._native.linear_tile(torch.empty(rows, depth, dtype=torch.float16, device="meta"), torch.tensor(widths), result32)


def test_the_wide_tile_is_taken_where_it_pays():
    """From 448 tiles on, up to 80 per cent of padding; not with a second round of a sixth or less, nor for results in fp32, where the
    tile of 64 features pads less."""
    assert _tile(56 * 256, 64, 1024) == (256, 128) and _tile(56 * 256 - 256, 64, 1024) == (128, 64)
    assert _tile(401408, 64, 64) == (256, 64) and _tile(401408, 64, 72) == (256, 128)
    # 512 tiles of two workgroups a CU: 513 to 597 of them
    assert _tile(171 * 256 - 256, 64, 320) == (256, 128) and _tile(171 * 256, 64, 320) == (256, 64) == _tile(199 * 256, 448, 320) and _tile(200 * 256, 64, 320) == (256, 128)
    assert _tile(104 * 256, 448, 320, 216) == (256, 64) and _tile(130 * 256, 448, 512) == (256, 128)
    assert _tile(200704, 192, 192) == _tile(200704, 192, 256, result32=1) == _tile(200704, 192, 320, result32=1) == (256, 128) != _tile(200704, 192, 192, result32=1)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("rows,depth,width", [(57601, 72, 264), (57400, 8, 144), (57345, 32, 256), (19201, 200, 776), (28800, 96, 512), (9000, 104, 1792)])
def test_wide_products_match_fp32(rows, depth, width, dtype):
    from dcnv4_amd import ext
    assert _tile(rows, depth, width) == (256, 128)
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


# 56 tiles of rows, the last one short, by 8 of both projections' features (320 and 540) and by 10 of the hidden ones (1280)
@pytest.mark.parametrize("dtype,tol", [(torch.float16, 3e-3), (torch.bfloat16, 2e-2)], ids=["fp16", "bf16"])      # as in test_gpu_layers.py
def test_layer_training_in_wide_products_matches_the_composition(dtype, tol):
    from dcnv4_amd.models.flash_intern_image import InternImageLayer
    torch.manual_seed(3)
    layer = InternImageLayer(320, 20, post_norm=True, layer_scale=0.3, dcn_output_bias=True, mlp_fc2_bias=True).cuda()
    with torch.no_grad():
        layer.dcn.offset_mask.weight.normal_(0, 0.02)
        layer.dcn.offset_mask.bias.normal_(0, 0.5)
    assert _tile(14310, 320, 320, 544) == _tile(14310, 320, 1280) == (256, 128)
    x, grad = torch.randn(2, 5, 2862, 320, device="cuda").unbind()
    results = []
    for run in (layer, lambda *a: _composed(layer, *a)):
        xi = x.clone().requires_grad_()
        with torch.autocast("cuda", dtype=dtype):
            out = run(xi, (54, 53))
        results.append([out.detach(), *torch.autograd.grad(out, [xi, *layer.parameters()], grad)])
    assert results[0][0].dtype == results[1][0].dtype
    for name, got, want in zip(["output", "x"] + [k for k, _ in layer.named_parameters()], *results):
        assert got.dtype == want.dtype and _rel(got, want) < tol, (name, _rel(got, want))
