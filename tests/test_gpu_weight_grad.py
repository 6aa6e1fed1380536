"""Weight gradients at the edges of their kernel: rows that fill no slice, fewer slices than buffers, splits that are short or
empty, both tiles in every type, columns that fill no tile."""
import pytest
import torch

from tests.test_gpu_layers import _composed, _rel

pytestmark = pytest.mark.gpu


LEVELS = [(128, 256), (64, 128), (1, 1)]
PIXELS = sum(h * w for h, w in LEVELS)
PLANS = {64: [(64, 54), (64, 64)], 256: [(128, 36), (128, 36)]}      # tile and splits, 16 bits and fp32


# rows: one slice and its remainders, two and three of them, four splits (the last one short); as many as the features, and then all
# products are one launch: the small tile with 54 splits (64 in fp32, the last ones empty), and the wide one with 36
@pytest.mark.parametrize("amp", [None, torch.float16, torch.bfloat16], ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("width,rows", [(64, 1), (64, 31), (64, 33), (128, 65), (256, 129), (256, 601), (64, PIXELS), (256, PIXELS)])
def test_weight_gradients_match_fp64(width, rows, amp):
    import dcnv4_amd
    from dcnv4_amd import ext
    torch.manual_seed(rows)
    heads = width // 32 if width > 64 else 4
    m = dcnv4_amd.FlashDeformAttn(width, 3, heads, 4).cuda()
    with torch.no_grad():           # locations that every type holds: the attention's output is the same in one call and in many
        m.sampling_offsets.weight.zero_()
        m.sampling_offsets.bias.copy_(torch.randint(-2, 3, m.sampling_offsets.bias.shape))
        m.attention_weights.weight.normal_(0, 0.05)
    shapes = torch.tensor(LEVELS, device="cuda")
    starts = torch.tensor([0, 128 * 256, 128 * 256 + 64 * 128], device="cuda")
    query, features = torch.randn(1, rows, width, device="cuda"), torch.randn(1, PIXELS, width, device="cuda")
    reference = torch.randint(0, 9, (1, rows, 3, 2), device="cuda") / 8
    grad = torch.randn(1, rows, width, device="cuda").to(amp or torch.float32)
    layers = [m.output_proj, m.sampling_offsets, m.value_proj, m.attention_weights]
    params = [p for layer in layers for p in (layer.weight, layer.bias)]
    if rows == PIXELS:
        plan = ext._native.weight_grad_plan(torch.empty(rows, width, dtype=amp or torch.float32, device="meta"),
                                            torch.tensor([layer.out_features for layer in layers]))
        assert plan == PLANS[width][amp is None]
    run = lambda: m(query, reference, features, shapes, starts)
    entered, left = [None] * 4, [None] * 4      # of each projection, where it runs by itself: what went in, the gradient of what came out

    def watch(i):
        def hook(module, args, out):
            entered[i] = args[0].detach()
            out.register_hook(lambda g: left.__setitem__(i, g))
        return layers[i].register_forward_hook(hook)

    with torch.autocast("cuda", dtype=amp or torch.float16, enabled=amp is not None):
        handles = [watch(i) for i in range(4)]
        torch.autograd.grad(run(), params, grad)
        for handle in handles:
            handle.remove()
        out = run()
    assert out.grad_fn.name() == "FlashDeformAttnBackward"
    got = torch.autograd.grad(out, params, grad)
    for i, layer in enumerate(layers):
        g, x = left[i].double().flatten(0, 1), entered[i].to(amp or torch.float32).double().flatten(0, 1)
        # the sums are in 32 bits, of products that 32 bits hold; what enters may differ by a rounding to the type, and by two behind the operator
        tol = {None: 1e-5, torch.float16: 1e-3, torch.bfloat16: 6e-3}[amp] * (1 if layer is m.output_proj else 2)
        print(f"{width} {rows} {amp} {i}: {_rel(got[2 * i], g.t() @ x):.2e} {_rel(got[2 * i + 1], g.sum(0)):.2e}")
        assert _rel(got[2 * i], g.t() @ x) < tol
        assert _rel(got[2 * i + 1], g.sum(0)) < (1e-6 if layer is m.output_proj else tol)


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
