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
    (64, 4, False, 3, 0.5, (40, 28, 28)), (512, 32, False, None, None, (1, 5, 7)), (272, 17, True, 3, 0.3, (1, 3, 11)),
    (640, 40, True, 3, 0.3, (1, 7, 7)), (48, 3, False, None, None, (42, 28, 29)), (112, 7, False, None, 0.5, (41, 28, 29)),
    (224, 14, True, 3, 0.3, (33, 32, 32))])
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


def _composed(layer, x, shape):
    """The layer run module by module: a forward hook on a child keeps the one-call path away."""
    handle = layer.mlp.register_forward_hook(lambda *a: None)
    try:
        return layer(x, shape)
    finally:
        handle.remove()


# channels, groups, post-norm, depthwise kernel, layer scale, (N, H, W), fp32 residual stream; 64- and 128-wide weight-gradient
# tiles with one split and several, rows that are no whole slice
TRAINING = [(64, 4, False, None, None, (3, 9, 7), False), (64, 4, False, 3, None, (2, 14, 11), True),
            (112, 7, True, 3, 0.3, (2, 17, 13), True), (160, 10, True, 5, None, (5, 7, 7), True),
            (112, 7, True, 3, 0.3, (13, 52, 50), True), (64, 4, False, None, None, (12, 28, 28), False)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("drop_path", [0.0, 0.4], ids=["no-drop", "drop-path"])
@pytest.mark.parametrize("channels,groups,post_norm,dw,scale,size,stream32", TRAINING, ids=[f"{c[0]}-{c[5][0]}x{c[5][1]}" for c in TRAINING])
def test_layer_training_under_autocast_matches_the_composition(channels, groups, post_norm, dw, scale, size, stream32, drop_path, dtype):
    from dcnv4_amd.models.flash_intern_image import InternImageLayer
    torch.manual_seed(channels + size[1])
    layer = InternImageLayer(channels, groups, post_norm=post_norm, layer_scale=scale, dw_kernel_size=dw, drop_path=drop_path,
                             dcn_output_bias=True, mlp_fc2_bias=True).cuda()
    with torch.no_grad():
        layer.dcn.offset_mask.weight.normal_(0, 0.02)
        layer.dcn.offset_mask.bias.normal_(0, 0.5)
        for name in ("gamma1", "gamma2"):
            if scale is not None:
                getattr(layer, name).uniform_(0.1, 0.5)
    n, h, w = size
    x = torch.randn(n, h * w, channels, device="cuda").to(torch.float32 if stream32 else dtype)
    grad = torch.randn_like(x)
    results = []
    for run in (layer, lambda *a: _composed(layer, *a)):
        torch.manual_seed(7)
        xi = x.clone().requires_grad_()
        with torch.autocast("cuda", dtype=dtype):
            out = run(xi, (h, w))
        grads = torch.autograd.grad(out, [xi, *layer.parameters()], grad)
        results.append([out.detach(), *grads])
    assert type(results[0]) is list and results[0][0].dtype == results[1][0].dtype
    tol = 3e-3 if dtype == torch.float16 else 2e-2
    names = ["output", "x"] + [k for k, _ in layer.named_parameters()]
    for name, got, want in zip(names, *results):
        assert got.dtype == want.dtype and got.shape == want.shape, name
        assert _rel(got, want) < tol, (name, _rel(got, want))


def test_layer_training_takes_one_node_and_reports_a_second_backward():
    from dcnv4_amd.models.flash_intern_image import InternImageLayer
    layer = InternImageLayer(64, 4).cuda()
    x = torch.randn(1, 64, 64, device="cuda", requires_grad=True)
    with torch.autocast("cuda", dtype=torch.float16):
        out = layer(x, (8, 8))
    assert out.grad_fn.name() == "InternImageLayerBackward"
    first = torch.autograd.grad(out.sum(), x, retain_graph=True)[0]
    assert torch.equal(first, torch.autograd.grad(out.sum(), x)[0])
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out.sum(), x)


# levels, queries (0: every pixel), reference coordinates, batch, padding, model width, points: few-row and tiled products, rows
# that fill no tile, feature rows that differ from query rows and do not
ATTENTION = [([(7, 9), (4, 5), (2, 3), (1, 2)], 0, 2, 3, True, 256, 4), ([(25, 31), (13, 16), (7, 8), (4, 4)], 77, 4, 2, True, 256, 4),
             ([(12, 10), (6, 5)], 33, 2, 1, False, 64, 8), ([(40, 52), (20, 26), (10, 13), (5, 7)], 0, 4, 2, False, 128, 4)]


@pytest.mark.parametrize("amp", [None, torch.float16, torch.bfloat16], ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("levels,queries,kind,batch,padded,width,points", ATTENTION, ids=[f"L{len(c[0])}-q{c[1]}-ref{c[2]}" for c in ATTENTION])
def test_attention_layer_in_one_call_matches_the_composition(levels, queries, kind, batch, padded, width, points, amp):
    import dcnv4_amd
    torch.manual_seed(queries + kind)
    m = dcnv4_amd.FlashDeformAttn(width, len(levels), 4, points).cuda()
    with torch.no_grad():
        m.sampling_offsets.weight.normal_(0, 0.05)
        m.attention_weights.weight.normal_(0, 0.05)
    pixels = sum(h * w for h, w in levels)
    q = queries or pixels
    shapes = torch.tensor(levels, device="cuda")
    starts = torch.tensor([sum(h * w for h, w in levels[:i]) for i in range(len(levels))], device="cuda")
    query, features = torch.randn(batch, q, width, device="cuda"), torch.randn(batch, pixels, width, device="cuda")
    reference = torch.rand(batch, q, len(levels), kind, device="cuda")
    mask = torch.rand(batch, pixels, device="cuda") < 0.2 if padded else None
    grad = torch.randn(batch, q, width, device="cuda").to(amp or torch.float32)
    results = []
    for composed in (False, True):
        handle = m.output_proj.register_forward_hook(lambda *a: None) if composed else None
        qi, fi = query.clone().requires_grad_(), features.clone().requires_grad_()
        with torch.autocast("cuda", dtype=amp or torch.float16, enabled=amp is not None):
            out = m(qi, reference, fi, shapes, starts, mask)
        assert (out.grad_fn.name() == "FlashDeformAttnBackward") != composed
        results.append([out.detach(), *torch.autograd.grad(out, [qi, fi, *m.parameters()], grad)])
        if composed:
            handle.remove()
    # fp32: a location that rounds to the other side in fp16 moves its sample
    tol = {None: 2e-3, torch.float16: 4e-3, torch.bfloat16: 2e-2}[amp]
    for name, got, want in zip(["output", "query", "features"] + [k for k, _ in m.named_parameters()], *results):
        assert got.dtype == want.dtype and got.shape == want.shape, name
        assert _rel(got, want) < tol, (name, _rel(got, want))
    if padded:
        assert not results[0][2][mask].any()


# either way of the gradient of value, whichever the sizes would take: by tiles the kernel that adds it up clears the padded rows
@pytest.mark.parametrize("scatter", ["tiled", "atomic"])
@pytest.mark.parametrize("amp", [None, torch.float16], ids=["fp32", "fp16"])
@pytest.mark.parametrize("queries,kind", [(0, 2), (0, 4), (50, 4)], ids=["pixels-ref2", "pixels-ref4", "few-ref4"])
def test_padded_rows_of_an_attention_layer_have_no_gradient(queries, kind, amp, scatter):
    import dcnv4_amd
    from dcnv4_amd import ext
    torch.manual_seed(kind)
    levels, batch, width = [(40, 52), (20, 26), (10, 13), (5, 7)], 2, 64
    m = dcnv4_amd.FlashDeformAttn(width, 4, 4, 4).cuda()
    with torch.no_grad():
        m.sampling_offsets.weight.normal_(0, 0.05)
        m.attention_weights.weight.normal_(0, 0.05)
    pixels = sum(h * w for h, w in levels)
    shapes = torch.tensor(levels, device="cuda")
    starts = torch.tensor([sum(h * w for h, w in levels[:i]) for i in range(4)], device="cuda")
    # a picture's right and lower edge in every level, and pixels here and there
    mask = torch.cat([((torch.arange(h)[:, None] >= 0.8 * h) | (torch.arange(w) >= 0.7 * w)).flatten() for h, w in levels]).expand(batch, -1).clone()
    mask = (mask & torch.tensor([[True], [False]])).cuda() | (torch.rand(batch, pixels, device="cuda") < 0.1)
    query, features = torch.randn(batch, queries or pixels, width, device="cuda"), torch.randn(batch, pixels, width, device="cuda")
    reference, grad = torch.rand(batch, queries or pixels, 4, kind, device="cuda"), torch.randn(batch, queries or pixels, width, device="cuda")
    results = []
    with ext.launch_options(scatter=scatter):
        value = torch.empty(batch, pixels, 4, width // 4, dtype=amp or torch.float32, device="meta")
        assert ext._native.attention_backward_tiled(value, 4, queries or pixels, 4) == (scatter == "tiled")
        for composed in (False, True):
            handle = m.output_proj.register_forward_hook(lambda *a: None) if composed else None
            qi, fi = query.clone().requires_grad_(), features.clone().requires_grad_()
            with torch.autocast("cuda", dtype=amp or torch.float16, enabled=amp is not None):
                out = m(qi, reference, fi, shapes, starts, mask)
            assert (out.grad_fn.name() == "FlashDeformAttnBackward") != composed
            results.append(torch.autograd.grad(out, [fi, m.value_proj.weight, m.value_proj.bias], grad.to(out.dtype)))
            if composed:
                handle.remove()
    for got, want in zip(*results):
        assert _rel(got, want) < (2e-3 if amp is None else 4e-3)      # as in the comparison with the composition above
    assert not results[0][0][mask].any() and results[0][0][~mask].any()


# products of few rows and of many
@pytest.mark.parametrize("amp", [None, torch.float16, torch.bfloat16], ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("h,w", [(6, 9), (64, 100)], ids=["few", "many"])
def test_query_gradient_in_fp32_is_two_products_added(h, w, amp):
    """One sum over both depths would be further from 64 bits.  With a query of zeros neither weight moves a point, so that the gradients
    of offsets and logits are the same whichever weight is zero: the gradient with both weights is the two with one of them, added."""
    import dcnv4_amd
    torch.manual_seed(h)
    m = dcnv4_amd.FlashDeformAttn(256, 1, 8, 4).cuda()
    shapes, starts = torch.tensor([[h, w]], device="cuda"), torch.zeros(1, dtype=torch.int64, device="cuda")
    features, reference = torch.randn(1, h * w, 256, device="cuda"), torch.rand(1, h * w, 1, 2, device="cuda")
    grad = torch.randn(1, h * w, 256, device="cuda")
    weights = [torch.randn_like(p.weight) for p in (m.sampling_offsets, m.attention_weights)]
    def query_gradient(*kept):
        with torch.no_grad():
            for p, weight, keep in zip((m.sampling_offsets, m.attention_weights), weights, kept):
                p.weight.copy_(weight * keep)
        query = torch.zeros(1, h * w, 256, device="cuda", requires_grad=True)
        with torch.autocast("cuda", dtype=amp or torch.float16, enabled=amp is not None):
            out = m(query, reference, features, shapes, starts)
        assert out.grad_fn.name() == "FlashDeformAttnBackward"
        return torch.autograd.grad(out, query, grad.to(out.dtype))[0]
    both, offsets, logits = query_gradient(1, 1), query_gradient(1, 0), query_gradient(0, 1)
    assert offsets.any() and logits.any() and torch.equal(both, logits + offsets)


# 16 queries of 54 pixels, and every pixel a query
@pytest.mark.parametrize("queries", [16, 54])
@pytest.mark.parametrize("amp", [None, torch.float16], ids=["fp32", "fp16"])
def test_attention_layer_trains_biases_of_frozen_weights(queries, amp):
    """The inputs, fp32 or the products' type, are kept for the weights' gradients only: biases do without."""
    import dcnv4_amd
    torch.manual_seed(0)
    m = dcnv4_amd.FlashDeformAttn(64, 1, 4, 4).cuda()
    shapes, starts = torch.tensor([[6, 9]], device="cuda"), torch.zeros(1, dtype=torch.int64, device="cuda")
    query, features = (torch.randn(2, n, 64, device="cuda", dtype=amp or torch.float32) for n in (queries, 54))
    reference, grad = torch.rand(2, queries, 1, 2, device="cuda"), torch.randn(2, queries, 64, device="cuda")

    def gradients(wanted):
        for p in m.parameters():
            p.requires_grad_(False)
        for p in wanted:
            p.requires_grad_(True)
        with torch.autocast("cuda", dtype=amp or torch.float16, enabled=amp is not None):
            out = m(query, reference, features, shapes, starts)
        assert out.grad_fn.name() == "FlashDeformAttnBackward"
        return torch.autograd.grad(out, wanted, grad.to(out.dtype))
    parameters = dict(m.named_parameters())
    every = dict(zip(parameters, gradients(list(parameters.values()))))
    biases = [name for name in parameters if name.endswith("bias")]
    for names in (biases, *([name] for name in biases)):
        for name, got in zip(names, gradients([parameters[name] for name in names])):
            assert _rel(got, every[name]) < (1e-5 if amp is None else 1e-3), name      # grad_value's terms come in an order that varies


@pytest.mark.parametrize("amp", [None, torch.float16], ids=["fp32", "fp16"])
def test_gradients_that_nobody_asked_for_have_memory_of_their_own(amp):
    """A frozen weight's gradient, formed with its bias's, is written by the last launch, which adds up the partial sums of all products:
    the gradients of feature rows, allocated behind those of query rows, may not lie in its memory."""
    import dcnv4_amd
    from dcnv4_amd import ext
    torch.manual_seed(0)
    m = dcnv4_amd.FlashDeformAttn(256, 1, 8, 4).cuda()
    with torch.no_grad():
        m.sampling_offsets.weight.normal_(0, 0.05)
        m.attention_weights.weight.normal_(0, 0.05)
    h, w, q = 32, 48, 1600
    shapes, starts = torch.tensor([[h, w]], device="cuda"), torch.zeros(1, dtype=torch.int64, device="cuda")
    query, features = torch.randn(1, q, 256, device="cuda"), torch.randn(1, h * w, 256, device="cuda")
    reference, grad = torch.rand(1, q, 1, 2, device="cuda"), torch.randn(1, q, 256, device="cuda")
    splits = ext._native.weight_grad_plan(torch.empty(q, 256, dtype=amp or torch.float32, device="meta"), torch.tensor([256, 64, 32]))[1]
    assert splits > 1      # so that there are partial sums of query rows

    def gradients(names):
        for name, p in m.named_parameters():
            p.requires_grad_(name in names)
        with torch.autocast("cuda", dtype=amp or torch.float16, enabled=amp is not None):
            out = m(query, reference, features, shapes, starts)
        assert out.grad_fn.name() == "FlashDeformAttnBackward"
        return dict(zip(names, torch.autograd.grad(out, [dict(m.named_parameters())[n] for n in names], grad.to(out.dtype))))
    every = [name for name, _ in m.named_parameters()]
    want = gradients(every)
    got = gradients([name for name in every if name.endswith("bias") or name.startswith("value_proj")])
    for name, g in got.items():
        assert _rel(g, want[name]) < (1e-5 if amp is None else 1e-3), name      # sums in fp32, grad_value's terms in an order that varies


def test_attention_layer_reads_changed_level_shapes_again():
    import dcnv4_amd
    m = dcnv4_amd.FlashDeformAttn(64, 1, 4, 4).cuda()
    shapes, starts = torch.tensor([[4, 6]], device="cuda"), torch.zeros(1, dtype=torch.int64, device="cuda")
    x, ref = torch.randn(1, 24, 64, device="cuda"), torch.rand(1, 24, 1, 2, device="cuda")
    with torch.no_grad():
        m(x, ref, x, shapes, starts)
        shapes[0, 0] = 5
        with pytest.raises(AssertionError, match="levels"):
            m(x, ref, x, shapes, starts)


@pytest.mark.parametrize("rows,depth,width", [(5, 16, 8), (129, 72, 104), (6000, 256, 384)])
def test_fp32_linear_matches_fp64(rows, depth, width):
    from dcnv4_amd import ext
    a, w, b = torch.randn(rows, depth, device="cuda"), torch.randn(width, depth, device="cuda"), torch.randn(width, device="cuda")
    product = a.double() @ w.double().t() + b.double()
    assert _rel(ext.linear_forward(a, w, b), product) < 1e-6
    assert _rel(ext.linear_forward(a, w, b, gelu=True), torch.nn.functional.gelu(product)) < 1e-6


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32], ids=["fp16", "bf16", "fp32"])
@pytest.mark.parametrize("rows", [3, 9000], ids=["few", "tiled"])
def test_gelu_epilogue_of_infinities_and_nan_is_the_frameworks(rows, dtype):
    from dcnv4_amd import ext
    a = torch.zeros(rows, 8, device="cuda", dtype=dtype)
    a[:3, 0] = torch.tensor([float("inf"), float("-inf"), float("nan")])
    w = torch.ones(64, 8, device="cuda", dtype=dtype)
    got = ext.linear_forward(a, w, gelu=True)[:3, 0]
    assert got.isnan().tolist() == [False, True, True] and got[0] == float("inf")
    assert torch.equal(got.isnan(), torch.nn.functional.gelu(a[:3, 0]).isnan())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
def test_gelu_epilogue_is_as_exact_as_the_fp32_function(dtype):
    """Every input of the type up to the end of its negative tail: the results' distance from 64 bits is no larger than that of the
    framework's function, which evaluates erf in fp32 and rounds once."""
    from dcnv4_amd import ext
    x = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dtype).cuda()
    x = x[(x.abs() < 13) & (x != 0)]
    a = torch.zeros(x.numel(), 8, device="cuda", dtype=dtype)
    a[:, 0] = x
    w = torch.zeros(8, 8, device="cuda", dtype=dtype)
    w[0, 0] = 1.0
    got = ext.linear_forward(a, w, gelu=True)[:, 0]
    exact = x.double() * torch.special.ndtr(x.double())
    framework = torch.nn.functional.gelu(x)
    assert _rel(got, exact) <= _rel(framework, exact)
    assert (got != exact.to(dtype)).sum() <= (framework != exact.to(dtype)).sum()


def test_fp32_bias_gradients_are_summed_by_slices():
    """Against 64 bits the framework's column sum over these rows is off by 2.3e-7 of its norm, a sum in slices of 32 rows by 2.0e-7,
    one running sum over each workgroup's rows by 6.5e-7."""
    import dcnv4_amd
    torch.manual_seed(0)
    m = dcnv4_amd.FlashDeformAttn(256, 1, 8, 4).cuda()
    h, w = 122, 250
    shapes, starts = torch.tensor([[h, w]], device="cuda"), torch.zeros(1, dtype=torch.int64, device="cuda")
    x, reference = torch.randn(1, h * w, 256, device="cuda"), torch.rand(1, h * w, 1, 2, device="cuda")
    grad = torch.randn(1, h * w, 256, device="cuda")
    out = m(x, reference, x, shapes, starts)
    assert out.grad_fn.name() == "FlashDeformAttnBackward"
    got = torch.autograd.grad(out, m.output_proj.bias, grad)[0]
    assert _rel(got, grad.double().sum((0, 1))) < 4e-7
