"""Calls of a handful of pixels: DCNv4's taps shared by the lanes of a quad, and the operator with its output projection in one kernel."""
import pytest
import torch

from tests.inputs import make_dcnv4_inputs
from tests.test_gpu_layers import _rel

pytestmark = pytest.mark.gpu


# up to 16384 vectors of 16 bytes a quad shares the taps, beyond it does not: one pixel, both sides of the edge, group widths of one to
# eight vectors, groups that do not fill a wave, images smaller than the kernel, dilation, an offset scale
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("B,H,W,G,D,dilation,scale", [(1, 1, 1, 1, 16, 1, 1.0), (1, 7, 7, 32, 16, 1, 1.0), (3, 5, 2, 7, 8, 2, 0.5), (1, 16, 16, 32, 16, 1, 1.0),
                                                      (1, 16, 16, 33, 16, 1, 1.0), (2, 9, 13, 5, 64, 1, 2.0)])
def test_forward_of_few_pixels_matches_the_direct_kernel(B, H, W, G, D, dilation, scale, dtype):
    from dcnv4_amd import ext
    value, rows, _ = (t.cuda().to(dtype) for t in make_dcnv4_inputs(B, H, W, G, D, seed=H * W + G))
    if G > 1:      # what is no number stays with its group; an infinite modulation is infinite, a point nowhere counts for nothing
        rows[0, 0, 0, 18], rows[0, 0, 0, 27 + 4], rows[0, -1, -1, 27 + 5] = float("inf"), float("nan"), float("-inf")
    call = lambda: ext.dcnv4_forward(value, rows, 3, 3, 1, 1, dilation, dilation, dilation, dilation, G, D, scale, 256, 0, 0, 0, False)
    got = call()
    with ext.launch_options(gather="direct"):
        want = call()
    # the same 36 products in fp32 in another order, rounded once
    bound = 36 * 2.0 ** -24 if dtype == torch.float32 else 2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7
    assert torch.equal(torch.isfinite(got), torch.isfinite(want))
    keep = torch.isfinite(want)
    assert _rel(got[keep], want[keep]) < bound


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("groups,shared", [(32, True), (33, False)])
def test_a_quad_shares_the_taps_of_up_to_16384_vectors(groups, shared, dtype):
    """Points on their pixels, values of 2^12: taps 0, 1 and 4 are 2^25, 1 and -2^25.  A lane of all nine loses the 1 next to 2^25; in a quad
    taps 0 and 4 are one lane's and cancel before another's 1 is added."""
    from dcnv4_amd import ext
    h, w = (16, 16) if dtype != torch.float32 else (8, 16)
    assert (h * w * groups * 16 * dtype.itemsize // 16 <= 16384) == shared
    value = torch.full((1, h, w, groups * 16), 2.0 ** 12, dtype=dtype, device="cuda")
    rows = torch.zeros(1, h, w, (groups * 27 + 7) // 8 * 8, dtype=dtype, device="cuda")
    taps = rows[..., :groups * 27].view(1, h, w, groups, 27)[..., 18:]
    taps[..., 0], taps[..., 1], taps[..., 4] = 2.0 ** 13, 2.0 ** -12, -2.0 ** 13
    out = ext.dcnv4_forward(value, rows, 3, 3, 1, 1, 1, 1, 1, 1, groups, 16, 1.0, 256, 0, 0, 0, False)
    assert (out[:, 1:-1, 1:-1] == (1 if shared else 0)).all()


# one round of workgroups and a round and a quarter of a workgroup's lanes at most: pixels in whole and ragged tiles, widths that are no
# multiple of 64, one vector a group and several, one pixel
LAYERS = [(16, 1, False, None, (1, 1, 1)), (64, 4, False, None, (1, 56, 56)), (64, 2, True, 0.3, (1, 33, 29)), (80, 5, True, 0.3, (1, 31, 33)),
          (128, 8, False, 0.5, (3, 13, 17)), (128, 4, True, 3.0, (1, 28, 28)), (256, 16, False, None, (1, 14, 14)), (320, 20, True, 0.3, (1, 14, 14)),
          (448, 7, False, None, (1, 5, 6)), (512, 32, False, 0.5, (1, 7, 7)), (640, 40, True, 0.3, (1, 7, 7)), (1024, 64, False, None, (1, 3, 4))]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("channels,groups,post_norm,scale,size", LAYERS, ids=[f"{c[0]}-{'post' if c[2] else 'pre'}" for c in LAYERS])
def test_layer_of_few_pixels_matches_the_modules_in_fp32(channels, groups, post_norm, scale, size, dtype):
    from dcnv4_amd import ext
    from dcnv4_amd.models.flash_intern_image import InternImageLayer
    torch.manual_seed(channels)
    layer = InternImageLayer(channels, groups, post_norm=post_norm, layer_scale=scale, dw_kernel_size=3 if post_norm else None,
                             dcn_output_bias=post_norm).cuda()
    with torch.no_grad():
        layer.dcn.offset_mask.weight.normal_(0, 0.02)
        layer.dcn.offset_mask.bias.normal_(0, 0.5)
    layer = layer.to(dtype).eval()
    n, h, w = size
    x = torch.randn(n, h * w, channels, device="cuda").to(dtype)
    assert ext._native.sampled_linear_fits(x, h, w, groups, 3)
    with torch.no_grad():
        got = layer(x, (h, w))
        want = layer.float()(x.float(), (h, w))
    tol = 2e-3 if dtype == torch.float16 else 1.5e-2      # a chain of roundings to the type, as in test_gpu_layers.py
    assert got.dtype == dtype and _rel(got, want) < tol
    assert _rel(got[-1, -1], want[-1, -1]) < 4 * tol and _rel(got[..., -8:], want[..., -8:]) < 2 * tol


def test_layer_of_few_pixels_sums_a_depth_in_eight_chains():
    """Eight chains, as many as products of few rows have: slices of 32 channels that are eight apart meet in one sum, where 2^25 and
    -2^25 are gone before the ones of the slices between are added.  The operator's points lie on their pixels and its values are the
    projection's biases, the MLP's are zero."""
    from dcnv4_amd import ext
    from dcnv4_amd.models.flash_intern_image import InternImageLayer
    layer = InternImageLayer(512, 32).cuda().half().eval()
    with torch.no_grad():
        for p in (layer.dcn.value_proj.weight, layer.dcn.offset_mask.weight, layer.dcn.offset_mask.bias, layer.dcn.output_proj.weight, layer.mlp.fc2.weight):
            p.zero_()
        layer.dcn.value_proj.bias.fill_(1.0)
        layer.dcn.value_proj.bias[0] = layer.dcn.value_proj.bias[8 * 32] = 2.0 ** 12
        layer.dcn.offset_mask.bias[:32 * 27].view(32, 27)[:, 18 + 4] = 1.0
        layer.dcn.output_proj.weight[:, 0], layer.dcn.output_proj.weight[:, 8 * 32] = 2.0 ** 13, -2.0 ** 13
        for slice in range(1, 8):
            layer.dcn.output_proj.weight[:, slice * 32] = 1.0
        x = torch.zeros(1, 49, 512, device="cuda", dtype=torch.float16)
        assert ext._native.sampled_linear_fits(x, 7, 7, 32, 3)
        assert (layer(x, (7, 7)) == 7.0).all()


def test_the_rule_of_the_kernel_for_few_pixels():
    from dcnv4_amd import ext
    fits = lambda n, h, w, c, kernel=3, dtype=torch.float16: ext._native.sampled_linear_fits(torch.empty(n, h * w, c, dtype=dtype, device="meta"), h, w, c // 16, kernel)
    assert fits(1, 64, 64, 64) and not fits(1, 64, 65, 64)              # 256 workgroups of 16 pixels
    assert fits(1, 14, 14, 256) and not fits(1, 14, 23, 256)            # 5 pixels a workgroup are a round and a quarter of its lanes, 6 are not
    assert not fits(1, 14, 14, 256, kernel=5) and not fits(1, 14, 14, 256, dtype=torch.float32) and not fits(1, 2, 2, 1040)


# tiles of 16 x 16 up to 320 of them: one element, ragged tiles, depths below a slice, that are no whole slice and beyond what a
# workgroup requests at once; 325 tiles go by 32 x 32
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("rows,width,depth", [(1, 8, 8), (17, 24, 40), (49, 512, 2048), (2, 96, 2088), (33, 40, 4168), (320, 256, 64), (400, 208, 64)])
def test_products_of_few_rows(rows, width, depth, dtype):
    from dcnv4_amd import ext
    torch.manual_seed(rows + depth)
    side = 32 if (rows, width) == (400, 208) else 16
    assert ext._native.linear_tile(torch.empty(rows, depth, dtype=dtype, device="meta"), torch.tensor([width]), 0) == (side, side)
    a, w, res = (torch.randn(*s, device="cuda").to(dtype) for s in ((rows, depth), (width, depth), (rows, width)))
    b, gamma = (torch.randn(width, device="cuda").to(dtype) for _ in range(2))
    product = a.double() @ w.double().t()
    # sums in fp32, of which a lane's chain has a sixteenth (fp32: a quarter), then one rounding of the result
    unit = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]
    assert _rel(ext.linear_forward(a, w), product) < unit + 1e-6
    assert _rel(ext.linear_forward(a, w, b, gamma, res), (product + b.double()) * gamma.double() + res.double()) < unit + 1e-6


def test_products_of_few_rows_add_their_parts_in_pairs():
    """Eight waves share a depth of 128 in fp32, sixteen elements each: their sums 2^25, 0, 2, 2, 1, 1, 1, 1 are exact in pairs; added one
    after the other all but the first are lost."""
    from dcnv4_amd import ext
    w = torch.zeros(8, 128, device="cuda")
    w[:, ::16] = torch.tensor([2.0 ** 25, 0.0, 2.0, 2.0, 1.0, 1.0, 1.0, 1.0], device="cuda")
    for rows in (1, 17):
        assert (ext.linear_forward(torch.ones(rows, 128, device="cuda"), w) == 2.0 ** 25 + 8).all()


# pixels x features in tiles of 16 x 16 (252 and 57 of them, the depth in one request and in two) and of 32 x 32 (1372 of 16 x 16): the
# depth is cut alike, so that results do not tell
@pytest.mark.parametrize("channels,size", [(112, (5, 15, 14)), (456, (1, 3, 5)), (112, (8, 28, 28))])
def test_downsampling_of_few_pixels(channels, size):
    from dcnv4_amd.models.flash_intern_image import DownsampleLayer
    torch.manual_seed(channels)
    n, h, w = size
    layer = DownsampleLayer(channels, "LN").cuda().half().eval()
    x = torch.randn(n, h * w, channels, device="cuda").half()
    with torch.no_grad():
        got, want = layer(x, (h, w)), layer.float()(x.float(), (h, w))
    assert got[1] == want[1] and _rel(got[0], want[0]) < 2e-3      # as in test_gpu_conv.py
