"""What a call through the extension module must not pass by: what torch's autograd Functions and modules refuse, record or let a
program replace, on the paths that run a whole operator or layer in one call."""
import gc

import pytest
import torch
import torch.autograd.forward_ad as fwAD

pytestmark = pytest.mark.gpu

GEOMETRY = (3, 3, 1, 1, 1, 1, 1, 1)
# A 16-bit intermediate rounds the other way where fp32 sums in front of it come in another order: a unit of its last place.
HALF_ULP = 2.0 ** -10


def _rel(got, want):
    return ((got.double() - want.double()).norm() / want.double().norm()).item()


def _layer(channels=64, dtype=torch.float16, **kw):
    from dcnv4_amd.models.flash_intern_image import InternImageLayer
    torch.manual_seed(channels)
    layer = InternImageLayer(channels, channels // 16, **kw).cuda()
    with torch.no_grad():
        layer.dcn.offset_mask.weight.normal_(0, 0.02)
        layer.dcn.offset_mask.bias.normal_(0, 0.5)
    return layer.to(dtype)


def _attention(width=64, levels=((6, 7), (3, 4)), queries=33, batch=2, module=None):
    import dcnv4_amd
    torch.manual_seed(queries)
    m = (module or dcnv4_amd.FlashDeformAttn)(width, len(levels), 4, 4).cuda()
    with torch.no_grad():
        m.sampling_offsets.weight.normal_(0, 0.05)
        m.attention_weights.weight.normal_(0, 0.05)
    pixels = sum(h * w for h, w in levels)
    shapes = torch.tensor(levels, device="cuda")
    starts = torch.tensor([sum(h * w for h, w in levels[:i]) for i in range(len(levels))], device="cuda")
    query, features = torch.randn(batch, queries, width, device="cuda"), torch.randn(batch, pixels, width, device="cuda")
    reference = torch.rand(batch, queries, len(levels), 2, device="cuda")
    return m, (query, reference, features, shapes, starts)


def _operators():
    """name -> (function of two float tensors, those tensors)"""
    from dcnv4_amd import DCNv4Function, FlashDeformAttnFunction
    from dcnv4_amd.functions import FlashDeformAttnSplitFunction
    rand = lambda *s: torch.randn(s, device="cuda")
    shapes, starts = torch.tensor([[5, 6], [3, 3]], device="cuda"), torch.tensor([0, 30], device="cuda")
    rows = torch.rand(1, 7, 2, 8 * 3, device="cuda")
    return {
        "dcnv4": (lambda v, o: DCNv4Function.apply(v, o, *GEOMETRY, 2, 16, 1.0, 256, 0), (rand(1, 6, 7, 32), rand(1, 6, 7, 56))),
        "attention": (lambda v, r: FlashDeformAttnFunction.apply(v, shapes, starts, r, 64, 4), (rand(1, 39, 2, 16), rows)),
        "attention split": (lambda v, r: FlashDeformAttnSplitFunction.apply(v, shapes, starts, r[..., :16].contiguous(), r[..., 16:].contiguous(), 64, 4),
                            (rand(1, 39, 2, 16), rows)),
    }


OPERATORS = ("dcnv4", "attention", "attention split")


def _poison():
    """Blocks that the allocator hands out next hold NaN."""
    torch.cuda.empty_cache()
    held = [torch.full((n,), float("nan"), device="cuda") for n in (64, 512, 4096, 65536, 1 << 20) for _ in range(32)]
    del held


@pytest.mark.parametrize("name", OPERATORS)
def test_a_traced_operator_computes_its_result(name):
    f, inputs = _operators()[name]
    traced = torch.jit.trace(f, inputs, check_trace=False)
    again = tuple(torch.rand_like(t) for t in inputs)
    _poison()
    assert torch.equal(traced(*again), f(*again))


@pytest.mark.parametrize("kind", ["inference", "autocast"])
def test_a_traced_layer_computes_its_result(kind):
    layer = _layer(dtype=torch.float16 if kind == "inference" else torch.float32).eval().requires_grad_(False)
    x, other = (torch.randn(2, 42, 64, device="cuda", dtype=layer.norm1[0].weight.dtype) for _ in range(2))

    def run(y):
        with torch.autocast("cuda", dtype=torch.float16, enabled=kind == "autocast"):
            return layer(y, (6, 7))

    with torch.no_grad():
        traced = torch.jit.trace(run, x, check_trace=False)
        _poison()
        assert _rel(traced(other), run(other)) < 3e-3


def test_a_traced_attention_layer_computes_its_result():
    m, (query, reference, features, shapes, starts) = _attention()
    m.requires_grad_(False)
    with torch.no_grad():
        traced = torch.jit.trace(lambda q, f: m(q, reference, f, shapes, starts), (query, features), check_trace=False)
        other = torch.randn_like(query), torch.randn_like(features)
        _poison()
        assert _rel(traced(*other), m(other[0], reference, other[1], shapes, starts)) < 2e-3


def test_a_traced_model_computes_its_result():
    from dcnv4_amd.models import flash_intern_image
    torch.manual_seed(1)
    model = flash_intern_image("t", depths=(1, 1, 1, 1)).cuda().half().eval()
    x, other = (torch.randn(1, 3, 64, 64, device="cuda").half() for _ in range(2))
    with torch.no_grad():
        traced = torch.jit.trace(model, x, check_trace=False)
        _poison()
        assert _rel(traced(other), model(other)) < 3e-3


class Wrapper(torch.Tensor):
    """Holds another tensor and has no storage of its own, as quantised or sharded parameters do."""

    @staticmethod
    def __new__(cls, held):
        return torch.Tensor._make_wrapper_subclass(cls, held.shape, dtype=held.dtype, device=held.device, requires_grad=False)

    def __init__(self, held):
        self.held = held

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        open_ = lambda t: t.held if isinstance(t, Wrapper) else t
        return func(*torch.utils._pytree.tree_map(open_, args), **torch.utils._pytree.tree_map(open_, kwargs or {}))


@pytest.mark.parametrize("kind", ["inference", "autocast", "attention"])
def test_parameters_without_storage_run_the_modules(kind):
    if kind == "attention":
        m, inputs = _attention()
        run, linear = lambda: m(*inputs), m.output_proj
    else:
        m = _layer(dtype=torch.float16 if kind == "inference" else torch.float32).eval()
        x = torch.randn(2, 42, 64, device="cuda", dtype=m.norm1[0].weight.dtype)
        run, linear = lambda: m(x, (6, 7)), m.mlp.fc1
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16, enabled=kind == "autocast"):
        want = run()
        linear._parameters["weight"] = Wrapper(linear.weight.detach())
        assert _rel(run(), want) < 3e-3


@pytest.mark.parametrize("kind", ["dcnv4", "layer", "attention"])
def test_gradients_without_storage_are_refused_and_zeros_are_zeros(kind):
    def forward():
        if kind == "dcnv4":
            f, (v, o) = _operators()["dcnv4"]
            return v.requires_grad_(), f(v, o)
        if kind == "attention":
            m, (x, *rest) = _attention()
            return x.requires_grad_(), m(x, *rest)
        x = torch.randn(2, 42, 64, device="cuda", requires_grad=True)
        with torch.autocast("cuda", dtype=torch.float16):
            return x, _layer(dtype=torch.float32)(x, (6, 7))

    x, out = forward()
    with pytest.raises(RuntimeError, match="memory"):
        torch.autograd.grad(out, x, Wrapper(torch.ones_like(out)))
    x, out = forward()
    zeros = torch._efficientzerotensor(out.shape, dtype=out.dtype, device="cuda")
    assert not torch.autograd.grad(out, x, zeros)[0].any()


@pytest.mark.parametrize("kind", ["post-norm", "pre-norm", "attention", "attention fp32"])
def test_a_gradient_may_begin_at_any_element(kind):
    if kind.startswith("attention"):
        m, (x, *rest) = _attention()
        run = lambda: m(x, *rest)
    else:
        m, x = _layer(dtype=torch.float32, post_norm=kind == "post-norm"), torch.randn(2, 42, 64, device="cuda")
        run = lambda: m(x, (6, 7))
    x.requires_grad_()
    with torch.autocast("cuda", dtype=torch.float16, enabled=kind != "attention fp32"):
        out = run()
    # as the split of a flattened cat hands it out
    shifted = torch.randn(out.numel() + 1, device="cuda").to(out.dtype)[1:].view(out.shape)
    assert shifted.is_contiguous() and shifted.data_ptr() % 16 != 0
    wanted = [x, *m.parameters()]
    got = torch.autograd.grad(out, wanted, shifted, retain_graph=True)
    for a, b in zip(got, torch.autograd.grad(out, wanted, shifted.clone())):
        assert _rel(a, b) < (1e-5 if kind == "attention fp32" else HALF_ULP)


@pytest.mark.parametrize("grad", [True, False], ids=["grad", "no-grad"])
@pytest.mark.parametrize("which", [0, 1])
@pytest.mark.parametrize("name", OPERATORS)
def test_an_operator_refuses_forward_mode(name, which, grad):
    f, inputs = _operators()[name]
    with fwAD.dual_level(), torch.set_grad_enabled(grad):
        inputs = list(inputs)
        inputs[which] = fwAD.make_dual(inputs[which], torch.ones_like(inputs[which]))
        with pytest.raises(NotImplementedError, match="jvp"):
            f(*inputs)


@pytest.mark.parametrize("where", ["input", "parameter"])
@pytest.mark.parametrize("kind", ["inference", "autocast", "attention"])
def test_a_layer_refuses_forward_mode(kind, where):
    if kind == "attention":
        m, (query, reference, features, shapes, starts) = _attention()
        run, x, weight = lambda q: m(q, reference, features, shapes, starts), query, m.value_proj
    else:
        m = _layer(dtype=torch.float16 if kind == "inference" else torch.float32).eval()
        x, weight = torch.randn(2, 42, 64, device="cuda", dtype=m.norm1[0].weight.dtype), m.dcn.value_proj
        run = lambda y: m(y, (6, 7))
    with fwAD.dual_level(), torch.no_grad(), torch.autocast("cuda", dtype=torch.float16, enabled=kind == "autocast"):
        if where == "input":
            x = fwAD.make_dual(x, torch.ones_like(x))
        else:
            w = weight.weight
            del weight.weight
            weight.register_parameter("weight", None)
            weight._parameters["weight"] = fwAD.make_dual(w.detach(), torch.ones_like(w))
        with pytest.raises(NotImplementedError, match="jvp"):
            run(x)


def test_the_convolutions_around_the_layers_carry_tangents():
    from dcnv4_amd.models.flash_intern_image import DownsampleLayer, StemLayer
    torch.manual_seed(2)
    stem, down = StemLayer(3, 64).cuda().half().eval(), DownsampleLayer(64).cuda().half().eval()
    x = torch.randn(1, 3, 32, 32, device="cuda").half()
    with torch.no_grad(), fwAD.dual_level():
        y = stem(fwAD.make_dual(x, torch.ones_like(x)))
        assert fwAD.unpack_dual(y).tangent is not None
        z, _ = down(y.reshape(1, 64, 64), (8, 8))
        assert fwAD.unpack_dual(z).tangent is not None


@pytest.mark.parametrize("kind", ["layer", "attention"])
def test_saved_tensor_hooks_see_the_activations(kind):
    if kind == "layer":
        m, x = _layer(dtype=torch.float32), torch.randn(2, 42, 64, device="cuda", requires_grad=True)
        run, least = lambda: m(x, (6, 7)), 2 * 42 * 64 * 8       # the hidden tensor before and after its activation
    else:
        m, (x, reference, features, shapes, starts) = _attention()
        x.requires_grad_()
        run, least = lambda: m(x, reference, features, shapes, starts), x.numel()
    wanted = [x, *m.parameters()]

    def grads():
        with torch.autocast("cuda", dtype=torch.float16, enabled=kind == "layer"):
            out = run()
        return torch.autograd.grad(out, wanted, torch.ones_like(out))

    seen = []
    plain = grads()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append((t.numel(), t.is_floating_point())) or t.cpu(), lambda t: t.cuda()):
        hooked = grads()
    assert sum(n for n, floating in seen if floating) > least + sum(p.numel() for p in m.parameters())
    for a, b in zip(plain, hooked):
        assert _rel(a, b) < 3e-3


def test_checkpointing_a_layer_frees_its_activations():
    from torch.utils.checkpoint import checkpoint
    layer, shape = _layer(dtype=torch.float32), (56, 56)
    x = torch.randn(4, 56 * 56, 64, device="cuda", requires_grad=True)

    def step(run):
        gc.collect()
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        with torch.autocast("cuda", dtype=torch.float16):
            out = run()
        kept = torch.cuda.memory_allocated() - before
        return kept, torch.autograd.grad(out, [x, *layer.parameters()], torch.ones_like(out))

    step(lambda: layer(x, shape))       # caches of the first call
    kept, want = step(lambda: layer(x, shape))
    held, got = step(lambda: checkpoint(layer, x, shape, use_reentrant=False))
    assert held < 2 * x.numel() * x.element_size() < kept       # the output and what torch keeps of small things
    for a, b in zip(want, got):
        assert _rel(b, a) < 3e-3


# the fused block tail takes a normalisation's parameters and calls its forward under autocast alone
@pytest.mark.parametrize("kind,child", [(k, c) for k in ("inference", "autocast") for c in ("mlp", "mlp.fc1", "mlp.act", "dcn", "dcn.value_proj")] +
                         [("autocast", "norm1.0")])
def test_a_replaced_forward_is_called(kind, child):
    layer = _layer(dtype=torch.float16 if kind == "inference" else torch.float32).eval()
    x = torch.randn(2, 42, 64, device="cuda", dtype=layer.norm1[0].weight.dtype)
    calls = []
    target = layer.get_submodule(child)
    forward = target.forward
    target.forward = lambda *a, **kw: calls.append(1) or forward(*a, **kw)
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16, enabled=kind == "autocast"):
        layer(x, (6, 7))
    assert calls == [1]


@pytest.mark.parametrize("child", ["value_proj", "output_proj"])
def test_a_replaced_forward_in_attention_is_called(child):
    m, inputs = _attention()
    calls, target = [], m.get_submodule(child)
    forward = target.forward
    target.forward = lambda *a: calls.append(1) or forward(*a)
    m(*inputs)
    assert calls == [1]


def test_replaced_forwards_around_the_layers_are_called():
    from dcnv4_amd.models.flash_intern_image import DownsampleLayer, StemLayer
    stem, down = StemLayer(3, 64).cuda().half().eval(), DownsampleLayer(64).cuda().half().eval()
    calls = []
    for m in (stem.conv1, stem.norm2, stem.norm2[0], down.norm, down.conv):
        m.forward = (lambda f: lambda *a: calls.append(1) or f(*a))(m.forward)
    with torch.no_grad():
        y = stem(torch.randn(1, 3, 32, 32, device="cuda").half())
        down(y.reshape(1, 64, 64), (8, 8))
    assert len(calls) == 5


@pytest.mark.parametrize("name", ["forward", "__call__"])
@pytest.mark.parametrize("cls", [torch.nn.GELU, torch.nn.Linear], ids=lambda c: c.__name__)
def test_a_class_with_a_replaced_method_is_called(cls, name, monkeypatch):
    layer, calls = _layer().eval(), []
    method = getattr(cls, name)
    monkeypatch.setattr(cls, name, lambda self, *a: calls.append(1) or method(self, *a))
    with torch.no_grad():
        layer(torch.randn(1, 42, 64, device="cuda").half(), (6, 7))
    assert len(calls) == (1 if cls is torch.nn.GELU else 5)


def test_subclasses_keep_what_they_override():
    import dcnv4_amd
    from dcnv4_amd.models.flash_intern_image import InternImageLayer
    calls = []

    class Centred(dcnv4_amd.FlashDeformAttn):
        def _sampling_locations(self, offsets, reference_points, spatial_shapes):
            calls.append("locations")
            return super()._sampling_locations(offsets, reference_points, spatial_shapes)

    m, inputs = _attention(module=Centred)
    m(*inputs)

    class Layer(InternImageLayer):
        def _scaled_norm(self, *a):
            calls.append("norm")
            return super()._scaled_norm(*a)

    layer = Layer(64, 4, post_norm=True).cuda().half().eval()
    with torch.no_grad():
        layer(torch.randn(1, 42, 64, device="cuda").half(), (6, 7))
    assert calls == ["locations", "norm", "norm"]


def test_wrapped_extension_functions_are_called(monkeypatch):
    from dcnv4_amd import ext
    calls = []
    for name in ("dcnv4_backward", "layer_norm_residual_forward", "depthwise_conv_forward"):
        f = getattr(ext, name)
        with monkeypatch.context() as patch:
            patch.setattr(ext, name, lambda *a, f=f, name=name, **kw: calls.append(name) or f(*a, **kw))
            layer = _layer(post_norm=True, dw_kernel_size=3, dtype=torch.float32 if name == "dcnv4_backward" else torch.float16)
            x = torch.randn(1, 42, 64, device="cuda", dtype=layer.norm1[0].weight.dtype)
            if name == "dcnv4_backward":
                with torch.autocast("cuda", dtype=torch.float16):
                    layer(x, (6, 7)).sum().backward()
            else:
                with torch.no_grad():
                    layer.eval()(x, (6, 7))
    assert set(calls) == {"dcnv4_backward", "layer_norm_residual_forward", "depthwise_conv_forward"}


def test_modes_and_subclasses_see_a_layers_operators():
    from torch.overrides import TorchFunctionMode
    from torch.utils.flop_counter import FlopCounterMode
    layer, x = _layer().eval(), torch.randn(1, 42, 64, device="cuda").half()
    products = 2 * 42 * 64 * (64 + 112 + 64 + 8 * 64)
    with torch.no_grad():
        with FlopCounterMode(display=False) as counter:
            layer(x, (6, 7))
        assert counter.get_total_flops() == products
        seen = []

        class Watch(TorchFunctionMode):
            def __torch_function__(self, func, types, args=(), kwargs=None):
                seen.append(func)
                return func(*args, **(kwargs or {}))

        with Watch():
            layer(x, (6, 7))
        assert torch.nn.functional.linear in seen

        class Named(torch.Tensor):
            pass

        assert type(layer(x.as_subclass(Named), (6, 7))) is Named


def test_a_default_device_keeps_the_one_call_path():
    layer, x = _layer(dtype=torch.float32), torch.randn(1, 42, 64, device="cuda")
    with torch.device("cuda"), torch.autocast("cuda", dtype=torch.float16):
        assert layer(x, (6, 7)).grad_fn.name() == "InternImageLayerBackward"


@pytest.mark.parametrize("kind", ["inference", "autocast", "attention"])
def test_a_plain_attribute_in_a_parameters_place_is_used(kind):
    if kind == "attention":
        m, inputs = _attention()
        run, linear = lambda: m(*inputs), m.output_proj
    else:
        m = _layer(dtype=torch.float16 if kind == "inference" else torch.float32).eval()
        x = torch.randn(2, 42, 64, device="cuda", dtype=m.norm1[0].weight.dtype)
        run, linear = lambda: m(x, (6, 7)), m.mlp.fc1
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16, enabled=kind == "autocast"):
        bias = torch.randn_like(linear.bias)
        linear.bias.copy_(bias)
        want = run()
        del linear.bias
        linear.bias = bias
        assert _rel(run(), want) < 3e-3


def _peak(f):
    gc.collect()        # modules of other tests that hold themselves
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    result = f()
    torch.cuda.synchronize()
    return torch.cuda.max_memory_allocated() - before, result


@pytest.mark.parametrize("kind", ["layer", "attention"])
def test_frozen_parameters_get_no_gradients_computed(kind):
    if kind == "layer":
        m, x = _layer(channels=512, dtype=torch.float32), torch.randn(1, 9, 512, device="cuda")
        run = lambda: m(x, (3, 3))
    else:
        m, (x, *rest) = _attention(width=512)
        run = lambda: m(x, *rest)
    x.requires_grad_()

    def backward(wanted):
        with torch.autocast("cuda", dtype=torch.float16):
            out = run()
        return _peak(lambda: torch.autograd.grad(out, wanted, torch.ones_like(out))[0])

    parameters = list(m.parameters())
    backward([x, *parameters])
    every, want = backward([x, *parameters])
    asked, _ = backward([x])          # the engine leaves the parameters' edges out
    m.requires_grad_(False)
    frozen, got = backward([x])
    assert max(frozen, asked) < every - 0.9 * 4 * sum(p.numel() for p in parameters) and _rel(got, want) < HALF_ULP


@pytest.mark.parametrize("kind", ["post-norm", "pre-norm", "attention"])
def test_each_gradient_alone_is_what_it_is_among_all(kind):
    if kind == "attention":
        m, (x, reference, features, *levels) = _attention()
        inputs, run = [x, features], lambda: m(x, reference, features, *levels)
    else:
        post = kind == "post-norm"
        m = _layer(dtype=torch.float32, post_norm=post, layer_scale=0.3 if post else None, dw_kernel_size=3, dcn_output_bias=True, mlp_fc2_bias=True)
        x = torch.randn(2, 42, 64, device="cuda")
        inputs, run = [x], lambda: m(x, (6, 7))
    wanted = [t.requires_grad_() for t in inputs] + list(m.parameters())
    with torch.autocast("cuda", dtype=torch.float16):
        out = run()
    grad = torch.randn_like(out)
    every = torch.autograd.grad(out, wanted, grad, retain_graph=True)
    for t, want in zip(wanted, every):
        assert _rel(torch.autograd.grad(out, t, grad, retain_graph=True)[0], want) < HALF_ULP


@pytest.mark.parametrize("kind", ["layer", "attention", "attention fp32"])
def test_a_forward_without_gradients_keeps_nothing_for_a_backward(kind):
    if kind == "layer":
        m, x = _layer(channels=256, dtype=torch.float32).eval(), torch.randn(2, 1024, 256, device="cuda")
        run, hidden = lambda: m(x, (32, 32)), 2 * 2 * 1024 * 1024
    else:
        m, inputs = _attention(width=512)
        run, hidden = lambda: m(*inputs), 0

    def forward():
        with torch.autocast("cuda", dtype=torch.float16, enabled=kind != "attention fp32"):
            return run()

    forward()
    with torch.no_grad():
        peak, got = _peak(forward)
    trained, want = _peak(forward)
    turned = (4 if kind == "attention fp32" else 2) * sum(p.numel() for p in m.parameters() if p.dim() == 2)
    assert peak <= trained - turned - hidden and torch.equal(got, want)


def test_the_gradient_of_a_pre_norm_layers_projections_meets_in_fp32():
    """The value projection's gradient is large and the same for all channels, which the normalisation's backward takes out; what is
    left came through the offsets and is small.  Added in 16 bits it would be lost in the rounding of the sum."""
    layer = _layer(dtype=torch.float32)
    with torch.no_grad():
        layer.dcn.value_proj.weight.copy_(32 * torch.randn(64, 1, device="cuda").expand(64, 64))
        layer.dcn.value_proj.bias.normal_()
        layer.mlp.fc2.weight.zero_()
    x, grad = torch.randn(2, 42, 64, device="cuda", requires_grad=True), torch.randn(2, 42, 64, device="cuda")

    def branch(amp):
        with torch.autocast("cuda", dtype=torch.float16, enabled=amp):
            out = layer(x, (6, 7))
        return torch.autograd.grad(out, x, grad)[0] - grad

    want = branch(False)
    got = branch(True)
    handle = layer.mlp.register_forward_hook(lambda *a: None)
    composed = branch(True)
    handle.remove()
    assert _rel(got, want) < 1.5 * _rel(composed, want)


def test_attention_layer_checks_shapes_written_past_the_version_counter():
    m, (query, reference, features, shapes, starts) = _attention()
    m(query, reference, features, shapes, starts)
    shapes.data[0, 0] = 7
    with pytest.raises(AssertionError, match="levels"):
        m(query, reference, features, shapes, starts)


def test_attention_layer_replays_from_a_graph():
    """The level check waits for the GPU and is left out of what a graph records; every replay reads the inputs as they are then."""
    m, (query, reference, features, shapes, starts) = _attention()
    m.requires_grad_(False)
    run = lambda: m(query, reference, features, shapes, starts)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        run()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = run()
    for _ in range(3):
        features.normal_()
        graph.replay()
        torch.cuda.synchronize()
        assert _rel(captured, run()) < 1e-6


def test_in_place_changes_after_a_layer_are_as_before():
    """What the composition does not save may change before the backward; what it saves may not."""
    layer = _layer(dtype=torch.float32, post_norm=True)
    x = torch.randn(1, 42, 64, device="cuda", requires_grad=True)
    with torch.autocast("cuda", dtype=torch.float16):
        stream = x * 1.0
        out = layer(stream, (6, 7))
        stream += 1.0
    want = torch.autograd.grad(out.sum(), x)
    m, (query, reference, features, shapes, starts) = _attention()
    q = query.clone().requires_grad_()
    out = m(q, reference, features, shapes, starts)
    reference.add_(1.0)
    torch.autograd.grad(out.sum(), q)
    out = m(q, reference, features, shapes, starts)
    with torch.no_grad():
        m.sampling_offsets.weight.add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(out.sum(), q)


def test_channels_last_models_keep_the_one_call_convolutions():
    from dcnv4_amd import ext
    from dcnv4_amd.models.flash_intern_image import DownsampleLayer, StemLayer
    torch.manual_seed(5)
    stem, down = StemLayer(3, 64).cuda().half().eval(), DownsampleLayer(64).cuda().half().eval()
    x, y = torch.randn(2, 3, 37, 30, device="cuda").half(), torch.randn(2, 35, 64, device="cuda").half()
    with torch.no_grad():
        want = stem(x), down(y, (5, 7))[0]
        stem, down = stem.to(memory_format=torch.channels_last), down.to(memory_format=torch.channels_last)
        got = ext._native.stem_inference(stem, x), ext._native.downsample_inference(down, y, 5, 7)
    assert all(g is not None and torch.equal(g, w) for g, w in zip(got, want))


def test_a_compiled_stem_is_one_graph_of_its_modules():
    from dcnv4_amd.models.flash_intern_image import DownsampleLayer, StemLayer
    torch.manual_seed(3)
    stem, down = StemLayer(3, 64).cuda().half().eval(), DownsampleLayer(64).cuda().half().eval()
    x, y = torch.randn(1, 3, 32, 32, device="cuda").half(), torch.randn(1, 64, 64, device="cuda").half()
    with torch.no_grad():
        assert _rel(torch.compile(stem, backend="eager", fullgraph=True)(x), stem(x)) < 2e-3
        assert _rel(torch.compile(down, backend="eager", fullgraph=True)(y, (8, 8))[0], down(y, (8, 8))[0]) < 2e-3


def test_a_layer_without_a_shape_takes_its_tokens_for_a_square():
    layer, x = _layer().eval(), torch.randn(1, 49, 64, device="cuda").half()
    with torch.no_grad():
        assert _rel(layer(x, None), layer(x, (7, 7))) < 3e-3


@pytest.mark.parametrize("kind", ["inference", "autocast"])
def test_settings_of_another_type_keep_their_value(kind):
    """What the operator's call converts to a number - a tensor of one element, a numpy integer - is no number to a reader of
    attributes."""
    import numpy as np
    layer = _layer(dtype=torch.float16 if kind == "inference" else torch.float32).eval()
    x = torch.randn(2, 42, 64, device="cuda", dtype=layer.norm1[0].weight.dtype)

    def run():
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16, enabled=kind == "autocast"):
            return layer(x, (6, 7))

    layer.dcn.offset_scale = 2.0
    want = run()
    layer.dcn.offset_scale = torch.tensor(2.0)
    assert _rel(run(), want) < 3e-3
    layer.dcn.offset_scale, layer.dcn.remove_center = 2.0, 1
    want = run()
    layer.dcn.remove_center = np.int64(1)
    assert _rel(run(), want) < 3e-3


def test_modules_added_to_a_sequential_run():
    from dcnv4_amd.models.flash_intern_image import DownsampleLayer, StemLayer, _norm
    torch.manual_seed(4)
    stem, down, layer = StemLayer(3, 64).cuda().half().eval(), DownsampleLayer(64).cuda().half().eval(), _layer(post_norm=True).eval()
    calls = []

    class Count(torch.nn.Module):
        def forward(self, x):
            calls.append(1)
            return x

    head = torch.nn.Sequential(torch.nn.Conv2d(64, 96, 1), _norm(96, "BN", "channels_first", "channels_first"), torch.nn.GELU()).cuda().half().eval()
    for sequential in (stem.norm1, stem.norm2, down.norm, layer.norm2, head, head[1]):
        sequential.add_module("extra", Count())
    from dcnv4_amd import ext
    with torch.no_grad():
        y = stem(torch.randn(1, 3, 32, 32, device="cuda").half()).reshape(1, 64, 64)
        down(y, (8, 8))
        layer(y, (8, 8))
        assert ext._native.head_inference(head, y, 8, 8) is None
    assert len(calls) == 4


@pytest.mark.parametrize("kind", ["layer", "attention"])
def test_a_node_lets_go_of_its_weights_after_the_backward(kind):
    """Weights that are no parameters - computed from others for one call - are held by nothing but the graph."""
    if kind == "layer":
        m, inputs, amp = _layer(channels=512, dtype=torch.float32), (torch.randn(1, 9, 512, device="cuda"), (3, 3)), True
    else:
        (m, inputs), amp = _attention(width=512), False
    values = {name: p.detach().clone() for name, p in m.named_parameters()}
    weights = {name: v.clone().requires_grad_() * 1.0 for name, v in values.items()}
    with torch.autocast("cuda", dtype=torch.float16, enabled=amp):
        out = torch.func.functional_call(m, weights, inputs)
    assert out.grad_fn.name() in ("InternImageLayerBackward", "FlashDeformAttnBackward")
    size = sum(w.numel() for w in weights.values() if w.dim() == 2) * 4
    gc.collect()
    before = torch.cuda.memory_allocated()
    out.sum().backward()
    del weights
    gc.collect()
    assert torch.cuda.memory_allocated() <= before - size and out.grad_fn is not None
