"""The convolutions around the layers in one call each - stem, downsampling, the head's 1 x 1 - against their modules in fp32: odd
sizes, a single output pixel, depths that end inside a slice, few rows and many, both memory formats of the picture."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rel(got, want):
    return ((got.double() - want.double()).norm() / want.double().norm()).item()


def _settled(module, dtype):
    """In eval mode with running statistics and affine parameters of its own."""
    for m in module.modules():
        if isinstance(m, torch.nn.BatchNorm2d):
            m.running_mean.normal_(0, 0.3)
            m.running_var.uniform_(0.5, 2.0)
        if isinstance(m, (torch.nn.BatchNorm2d, torch.nn.LayerNorm)):
            torch.nn.init.normal_(m.weight, 1.0, 0.2)
            torch.nn.init.normal_(m.bias, 0.0, 0.2)
    return module.cuda().to(dtype).eval()


@pytest.mark.parametrize("dtype,tol", [(torch.float16, 2e-3), (torch.bfloat16, 1.5e-2)], ids=["fp16", "bf16"])
@pytest.mark.parametrize("channels,size", [(64, (1, 3, 3)), (80, (2, 37, 51)), (112, (3, 64, 33)), (192, (1, 40, 20)), (64, (20, 224, 160))])
@pytest.mark.parametrize("layout", [torch.contiguous_format, torch.channels_last], ids=["nchw", "nhwc"])
def test_stem_matches_its_modules_in_fp32(channels, size, layout, dtype, tol):
    from dcnv4_amd.models.flash_intern_image import StemLayer
    torch.manual_seed(channels)
    stem = _settled(StemLayer(3, channels, "BN"), dtype)
    n, h, w = size
    x = torch.randn(n, 3, h, w, device="cuda").to(dtype).contiguous(memory_format=layout)
    with torch.no_grad():
        got = stem(x)
        want = stem.float()(x.float())
    assert got.dtype == dtype and got.shape == want.shape and got.is_contiguous() and _rel(got, want) < tol


@pytest.mark.parametrize("dtype,tol", [(torch.float16, 2e-3), (torch.bfloat16, 1.5e-2)], ids=["fp16", "bf16"])
@pytest.mark.parametrize("channels,size", [(8, (1, 1, 1)), (64, (1, 7, 9)), (112, (5, 15, 14)), (448, (2, 14, 14)), (256, (1, 14, 14)), (64, (24, 56, 57)),
                                           (136, (40, 29, 30))])
def test_downsampling_matches_its_modules_in_fp32(channels, size, dtype, tol):
    from dcnv4_amd.models.flash_intern_image import DownsampleLayer
    torch.manual_seed(channels)
    layer = _settled(DownsampleLayer(channels), dtype)
    n, h, w = size
    x = torch.randn(n, h * w, channels, device="cuda").to(dtype)
    with torch.no_grad():
        got, shape = layer(x, (h, w))
        want, want_shape = layer.float()(x.float(), (h, w))
    assert shape == want_shape and got.dtype == dtype and got.shape == want.shape and _rel(got, want) < tol


# Wide tiles (256 pixels x 128 features, at least 288 of them): a last tile of 232 pixels and a depth of 45 vectors in slices of four;
# a second tile of 16 features; channels that straddle lines; whole tiles of whole lines.  The convolution's result and the
# normalisation's are rounded once each to the type: within two units of roundoff.
@pytest.mark.parametrize("dtype,unit", [(torch.float16, 2.0**-11), (torch.bfloat16, 2.0**-8)], ids=["fp16", "bf16"])
@pytest.mark.parametrize("channels,size", [(40, (24, 113, 110)), (72, (12, 111, 113)), (120, (13, 106, 107)), (64, (96, 56, 56))])
def test_wide_downsampling_matches_its_modules_in_fp32(channels, size, dtype, unit):
    from dcnv4_amd.models.flash_intern_image import DownsampleLayer
    torch.manual_seed(channels)
    layer = _settled(DownsampleLayer(channels), dtype)
    n, h, w = size
    x = torch.randn(n, h * w, channels, device="cuda").to(dtype)
    with torch.no_grad():
        got, _ = layer(x, (h, w))
        want, _ = layer.float()(x.float(), (h, w))
    assert _rel(got, want) < 2 * unit


@pytest.mark.parametrize("rows", [1, 49, 5000])
def test_the_heads_convolution_matches_its_modules_in_fp32(rows):
    from dcnv4_amd import ext
    from dcnv4_amd.models.flash_intern_image import _norm
    head = _settled(torch.nn.Sequential(torch.nn.Conv2d(120, 200, 1, bias=False), _norm(200, "BN", "channels_first", "channels_first"), torch.nn.GELU()),
                    torch.float16)
    x = torch.randn(2, rows, 120, device="cuda").half()
    with torch.no_grad():
        got = ext._native.head_inference(head, x, rows, 1)
        want = head.float()(x.float().permute(0, 2, 1)[..., None])[..., 0].permute(0, 2, 1)
    assert _rel(got.view(2, rows, 200), want) < 2e-3
