"""The matrix-core linear kernels at the edges of their tiles, and a FlashInternImage layer's one-call inference against the
composition of its modules in fp32."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rel(got, want):
    return ((got.double() - want.double()).norm() / want.double().norm()).item()


# rows x depth x width: few rows (one fragment, a ragged tile, a deep product), 64 / 128 / 256-row tiles with a remainder in every
# direction, a depth that is not a whole slice
LINEAR = [(1, 8, 8), (33, 72, 40), (49, 2048, 512), (500, 64, 96), (1000, 112, 760), (3137, 256, 64), (9000, 120, 448), (40001, 112, 192),
          (70000, 64, 520)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("rows,depth,width", LINEAR, ids=lambda v: str(v))
def test_linear_with_its_epilogues_matches_fp32(rows, depth, width, dtype):
    from dcnv4_amd import ext
    g = torch.Generator(device="cuda").manual_seed(rows)
    rand = lambda *shape: torch.randn(shape, generator=g, device="cuda").to(dtype)
    a, w, b, gamma, res = rand(rows, depth), rand(width, depth) / depth ** 0.5, rand(width), rand(width), rand(rows, width)
    tol = 1e-3 if dtype == torch.float16 else 6e-3
    product = a.float() @ w.float().t()
    assert _rel(ext.linear_forward(a, w), product) < tol
    want = torch.nn.functional.gelu(product + b.float())
    assert _rel(ext.linear_forward(a, w, b, gelu=True), want) < tol
    assert _rel(ext.linear_forward(a, w, b, gamma, res, gelu=True), want * gamma.float() + res.float()) < tol


def test_gelu_epilogue_keeps_its_relative_precision_in_the_tails():
    from dcnv4_amd import ext
    x = torch.linspace(-5.0, 6.0, 4096, device="cuda").half()
    a = torch.zeros(4096, 8, device="cuda", dtype=torch.float16)
    a[:, 0] = x
    w = torch.zeros(8, 8, device="cuda", dtype=torch.float16)
    w[0, 0] = 1.0
    got = ext.linear_forward(a, w, gelu=True)[:, 0].double()
    want = torch.nn.functional.gelu(x.double())
    assert ((got - want).abs() <= 5.5e-4 * want.abs() + 6e-8).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("channels,groups,post_norm,dw,scale,size", [
    (64, 4, False, None, None, (3, 13, 9)), (112, 7, True, 3, 0.3, (2, 14, 11)), (160, 10, True, 5, None, (1, 7, 7)),
    (64, 4, False, 3, 0.5, (40, 28, 28))])
def test_layer_inference_matches_the_modules_in_fp32(channels, groups, post_norm, dw, scale, size, dtype):
    from dcnv4_amd.models.flash_intern_image import InternImageLayer
    torch.manual_seed(channels)
    layer = InternImageLayer(channels, groups, post_norm=post_norm, layer_scale=scale, dw_kernel_size=dw, drop=0.1, drop_path=0.1).cuda()
    with torch.no_grad():
        layer.dcn.offset_mask.weight.normal_(0, 0.02)
        layer.dcn.offset_mask.bias.normal_(0, 0.5)
    layer = layer.to(dtype).eval()
    n, h, w = size
    x = torch.randn(n, h * w, channels, device="cuda").to(dtype)
    with torch.no_grad():
        assert layer.dcn.center_feature_scale is False
        got = layer(x, (h, w))
        seen = []
        handle = layer.mlp.register_forward_hook(lambda *a: seen.append(1))      # a hooked layer runs its modules
        composed = layer(x, (h, w))
        handle.remove()
        want = layer.float()(x.float(), (h, w))
    assert seen == [1] and got.dtype == dtype
    tol = 2e-3 if dtype == torch.float16 else 1.5e-2
    assert _rel(got, want) < tol and _rel(composed, want) < tol
