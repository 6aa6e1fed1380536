"""Weight gradients at the edges of their kernel: rows that fill no slice, fewer slices than buffers, splits that are short or
empty, both tiles in every type, columns that fill no tile."""
import pytest
import torch

from tests.test_gpu_layers import _composed, _rel

pytestmark = pytest.mark.gpu


LEVELS = [(128, 256), (64, 128), (1, 1)]
PIXELS = sum(h * w for h, w in LEVELS)


# rows: one slice and its remainders, two and three of them, four splits (the last one short); as many as the features, and then all
# products are one launch: the small tile with 54 splits (64 in fp32, the last ones empty), the wide one with 32 (36)
@pytest.mark.parametrize("amp", [None, torch.float16, torch.bfloat16], ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("width,rows", [(64, 1), (64, 31), (64, 33), (128, 65), (256, 129), (256, 601), (64, PIXELS), (256, PIXELS)])
def test_weight_gradients_match_fp64(width, rows, amp):
    import dcnv4_amd
    torch.manual_seed(rows)
    m = dcnv4_amd.FlashDeformAttn(width, 3, width // 32 if width > 64 else 4, 4).cuda()
    with torch.no_grad():           # locations that every type holds: the attention's output is the same in one call and in many
        m.sampling_offsets.weight.zero_()
        m.sampling_offsets.bias.copy_(torch.randint(-2, 3, m.sampling_offsets.bias.shape))
        m.attention_weights.weight.normal_(0, 0.05)
    shapes = torch.tensor(LEVELS, device="cuda")
    starts = torch.tensor([0, 128 * 256, 128 * 256 + 64 * 128], device="cuda")
    query, features = torch.randn(1, rows, width, device="cuda"), torch.randn(1, PIXELS, width, device="cuda")
    reference = torch.randint(0, 9, (1, rows, 3, 2), device="cuda") / 8
    grad = torch.randn(1, rows, width, device="cuda").to(amp or torch.float32)
    run = lambda: m(query, reference, features, shapes, starts)
    seen = []
    with torch.autocast("cuda", dtype=amp or torch.float16, enabled=amp is not None):
        handle = m.output_proj.register_forward_hook(lambda module, args, out: seen.append(args[0].detach()))
        run()
        handle.remove()
        out = run()
    assert out.grad_fn.name() == "FlashDeformAttnBackward"
    got_w, got_b = torch.autograd.grad(out, [m.output_proj.weight, m.output_proj.bias], grad)
    g, x = grad.double().flatten(0, 1), seen[0].to(amp or torch.float32).double().flatten(0, 1)
    # the sums are in 32 bits, of products that 32 bits hold; what enters may differ by a rounding to the type
    tol = {None: 1e-5, torch.float16: 1e-3, torch.bfloat16: 6e-3}[amp]
    assert _rel(got_w, g.t() @ x) < tol and _rel(got_b, g.sum(0)) < 1e-6


# 80, 160 and 448 channels: 128-wide tiles of 51, 12 and 3 splits
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("channels,groups,size", [(80, 5, (5, 124, 124)), (160, 10, (1, 139, 139)), (448, 28, (3, 40, 41)), (64, 4, (1, 3, 11))])
def test_layer_weight_gradients_in_wide_tiles_match_the_composition(channels, groups, size, dtype):
    from dcnv4_amd.models.flash_intern_image import InternImageLayer
    torch.manual_seed(channels)
    layer = InternImageLayer(channels, groups, post_norm=True, dw_kernel_size=3, dcn_output_bias=True, mlp_fc2_bias=True).cuda()
    with torch.no_grad():
        layer.dcn.offset_mask.weight.normal_(0, 0.02)
        layer.dcn.offset_mask.bias.normal_(0, 0.5)
    n, h, w = size
    x = torch.randn(n, h * w, channels, device="cuda").to(dtype)
    grad, weights = torch.randn_like(x) / 64, [p for p in layer.parameters() if p.dim() == 2]
    results = []
    for run in (layer, lambda *a: _composed(layer, *a)):
        with torch.autocast("cuda", dtype=dtype):
            out = run(x.clone().requires_grad_(), (h, w))
        results.append(torch.autograd.grad(out, weights, grad))
    for got, want in zip(*results):      # the modules' gradients pass through the type
        assert _rel(got, want) < (3e-3 if dtype == torch.float16 else 2e-2)
