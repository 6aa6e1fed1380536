"""Calls of a handful of pixels: DCNv4's taps shared by the lanes of a quad."""
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
