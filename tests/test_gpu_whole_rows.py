"""Layers whose products are normalised before they leave their kernel (rows enough to fill the chip): widths at every edge of a wave's
share of the features, a ragged last tile of rows, depths that are no whole slice, with and without layer scale and biases, the
normalisation in front of the residual and behind it, alone and behind the one-kernel MLP.  Against the modules in fp32.  And the rule
at its edges: the shapes below are taken by that kernel, each width of a wave's share of the features among them."""
import pytest
import torch

from tests.test_gpu_layers import _rel

pytestmark = pytest.mark.gpu

# channels, groups, post-norm, depthwise kernel, layer scale, (N, H, W), MLP ratio
LAYERS = [(48, 3, True, None, None, (42, 28, 29), 4.0), (64, 4, True, 3, 0.3, (17, 31, 33), 4.0), (80, 5, False, None, 0.5, (21, 28, 29), 2.0),
          (144, 9, True, None, 0.3, (43, 20, 41), 4.0), (144, 9, False, 3, None, (17, 31, 33), 1.0), (176, 11, True, 3, None, (21, 31, 33), 3.0),
          (256, 16, True, None, 0.3, (21, 31, 33), 1.0), (256, 16, False, None, None, (25, 31, 33), 2.0),
          (320, 20, True, 3, 0.3, (129, 14, 14), 1.0), (320, 20, False, None, 0.5, (129, 14, 14), 1.0), (368, 23, True, None, None, (129, 14, 14), 1.0),
          (368, 23, False, 3, 0.5, (129, 14, 14), 1.0), (448, 28, True, None, 0.3, (129, 14, 14), 1.0), (448, 28, False, None, None, (129, 14, 14), 1.0),
          (512, 32, False, None, None, (129, 14, 14), 1.0), (512, 32, True, 3, 0.3, (129, 14, 14), 1.0)]


# workgroups of 128 rows: half and five eighths of the 256 CUs, three quarters of them; three fifths with one to a CU; six sevenths of two rounds
@pytest.mark.parametrize("width,after_residual,least", [(8, 0, 128), (160, 1, 128), (168, 0, 160), (256, 0, 160), (168, 1, 192), (256, 1, 192),
                                                        (264, 0, 154), (512, 1, 154)])
def test_the_kernel_is_taken_from_enough_workgroups_on(width, after_residual, least):
    from dcnv4_amd import ext
    takes = lambda workgroups, dtype=torch.float16, n=width: ext._native.rows_fits(torch.empty(workgroups * 128 - 7, 64, dtype=dtype, device="meta"), n, after_residual)
    assert takes(least) and takes(least, torch.bfloat16) and not takes(least - 1)
    assert takes(257) == (width <= 256) and takes(439) and takes(438) == (width <= 256) and not takes(512, n=520)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("channels,groups,post_norm,dw,scale,size,ratio", LAYERS, ids=[f"{c[0]}-{'post' if c[2] else 'pre'}" for c in LAYERS])
def test_layer_of_many_rows_matches_the_modules_in_fp32(channels, groups, post_norm, dw, scale, size, ratio, dtype):
    from dcnv4_amd.models.flash_intern_image import InternImageLayer
    torch.manual_seed(channels)
    layer = InternImageLayer(channels, groups, post_norm=post_norm, layer_scale=scale, dw_kernel_size=dw, mlp_ratio=ratio,
                             dcn_output_bias=post_norm, mlp_fc2_bias=post_norm).cuda()
    with torch.no_grad():
        layer.dcn.offset_mask.weight.normal_(0, 0.02)
        layer.dcn.offset_mask.bias.normal_(0, 0.5)
        for norm in (layer.norm1, layer.norm2):
            norm[0].weight.uniform_(0.5, 1.5)
            norm[0].bias.normal_(0, 0.3)
    layer = layer.to(dtype).eval()
    n, h, w = size
    x = torch.randn(n, h * w, channels, device="cuda").to(dtype)
    from dcnv4_amd import ext
    assert ext._native.rows_fits(x, channels, not post_norm)
    with torch.no_grad():
        got = layer(x, (h, w))
        want = layer.float()(x.float(), (h, w))
    tol = 2e-3 if dtype == torch.float16 else 1.5e-2      # a chain of roundings to the type, as in test_gpu_layers.py
    assert got.dtype == dtype and _rel(got, want) < tol
    # the last rows, and the last features, by themselves
    assert _rel(got[-1, -70:], want[-1, -70:]) < 2 * tol and _rel(got[..., -8:], want[..., -8:]) < 2 * tol
