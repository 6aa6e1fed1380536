"""The workloads by which this framework's speed is judged, as its users run them: the DCNv4 operator and flash
deformable attention through their autograd Functions, the layers built on them, and FlashInternImage itself.

A case is a dict of plain values; ``prepare`` makes what a program has in hand before the call, ``run`` is one pass.
The kinds:

  dcnv4            DCNv4Function on an NHWC image and its packed offset rows
  attention        FlashDeformAttnFunction on packed (locations, logits) rows
  attention_layer  the FlashDeformAttn module (projections, locations, sampling), training
  block            one FlashInternImage layer (DCNv4 module, block tails, MLP), training under autocast
  model            FlashInternImage in eval mode, 16-bit weights: images to logits
"""
import math

import torch

from dcnv4_amd import DCNv4Function, FlashDeformAttn, FlashDeformAttnFunction
from dcnv4_amd.models import flash_intern_image
from dcnv4_amd.models.flash_intern_image import InternImageLayer

_DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
_LEVELS = 4            # pyramid levels of the attention cases, each half of the one before
_HEADS, _HEAD_WIDTH, _POINTS = 8, 32, 4
_DEPTHS = {"t": (4, 4, 18, 4), "s": (4, 4, 21, 4), "b": (4, 4, 21, 4)}
_CHANNELS = {"t": 64, "s": 80, "b": 112}


def listed():
    def dcnv4(name, batch, height, width, groups, group_width, dtype, train, offsets="uniform", spread=3.0):
        return dict(name=name, kind="dcnv4", batch=batch, height=height, width=width, groups=groups, group_width=group_width,
                    dtype=dtype, train=train, offsets=offsets, spread=spread)

    return [
        # one image at the last stage of FlashInternImage-T: the smallest call, what a request of batch 1 consists of
        dcnv4("dcnv4 fwd 1x7x7 fp16", 1, 7, 7, 32, 16, "float16", False),
        # training of FlashInternImage-T at 224 pixels, batch 64: its largest stage in half precision
        dcnv4("dcnv4 train 64x56x56 fp16", 64, 56, 56, 4, 16, "float16", True),
        # and the stage that holds 18 of its 30 layers, in single precision
        dcnv4("dcnv4 train 64x14x14 fp32", 64, 14, 14, 16, 16, "float32", True),
        # serving of FlashInternImage-B in batches of 128: first stage, an odd number of groups
        dcnv4("dcnv4 fwd 128x56x56 fp16", 128, 56, 56, 7, 16, "float16", False),
        # a detector's training at 800 x 1333 pixels, two images: first stage of the L variant, a ragged width, learnt
        # offsets with tails rather than a bounded range
        dcnv4("dcnv4 train 2x200x334 bf16", 2, 200, 334, 10, 16, "bfloat16", True, "normal", 2.0),
        # few wide groups (64 channels), one of the launch keys the operator is tuned for
        dcnv4("dcnv4 train 64x28x28 wide", 64, 28, 28, 4, 64, "float16", True),
        # attention inference in a deformable encoder: every pixel of a 128 x 128 pyramid is a query, 4 images
        dict(name="attention fwd 4x128x128 fp16", kind="attention", batch=4, height=128, width=128, queries=0,
             dtype="float16", train=False),
        # encoder layer of a detector in training: two padded images of 800 x 1216 pixels, single precision
        dict(name="encoder train 2x100x152 fp32", kind="attention_layer", batch=2, height=100, width=152, queries=0,
             amp="none", boxes=False),
        # decoder layer of the same detector with refined boxes as reference, 300 queries, mixed precision
        dict(name="decoder train 2x300 amp", kind="attention_layer", batch=2, height=100, width=152, queries=300,
             amp="float16", boxes=True),
        # a layer of FlashInternImage-B's third stage in mixed-precision training, batch 64
        dict(name="block train 64x14x14 amp", kind="block", batch=64, height=14, width=14, channels=448, groups=28,
             post_norm=True, amp="float16"),
        # one picture through FlashInternImage-T: latency
        dict(name="model t 1x224 fp16", kind="model", variant="t", batch=1, image=224, dtype="float16"),
        # throughput of FlashInternImage-B in batches of 128
        dict(name="model b 128x224 fp16", kind="model", variant="b", batch=128, image=224, dtype="float16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_one(rng):
    kind = rng.choices(("dcnv4", "attention", "attention_layer", "block", "model"), (8, 2, 3, 4, 3))[0]
    if kind == "dcnv4":
        offsets = rng.choice(("uniform", "normal"))
        case = dict(kind=kind, batch=_log_int(rng, 1, 128), height=_log_int(rng, 7, 256), width=_log_int(rng, 7, 334),
                    groups=_log_int(rng, 1, 80), group_width=rng.choice((16, 16, 16, 32, 64)),
                    dtype=rng.choice(tuple(_DTYPES)), train=rng.random() < 0.6, offsets=offsets,
                    spread=round(rng.uniform(1.0, 4.0) if offsets == "uniform" else rng.uniform(0.5, 2.0), 2))
        elements = case["batch"] * case["height"] * case["width"] * case["groups"] * case["group_width"]
        return case if 25_000 <= elements <= 45_000_000 else None
    if kind in ("attention", "attention_layer"):
        case = dict(kind=kind, batch=_log_int(rng, 1, 8), height=_log_int(rng, 24, 160), width=_log_int(rng, 24, 160),
                    queries=0 if rng.random() < 0.5 else _log_int(rng, 100, 900))
        if kind == "attention":
            case.update(dtype=rng.choice(("float32", "float16")), train=rng.random() < 0.5)
        else:
            case.update(amp=rng.choice(("none", "float16")), boxes=case["queries"] > 0 and rng.random() < 0.5)
        return case if case["batch"] * _pyramid(case)[1] <= 90_000 else None
    if kind == "block":
        stage = rng.randrange(4)
        variant = rng.choice(("t", "s", "b"))
        size = rng.uniform(0.7, 2.5) * 56 / 2 ** stage
        channels = _CHANNELS[variant] * 2 ** stage
        case = dict(kind=kind, batch=_log_int(rng, 1, 128), height=max(4, int(size)), width=max(4, int(size * rng.uniform(0.8, 1.5))),
                    channels=channels, groups=channels // 16, post_norm=variant != "t", amp=rng.choice(("float16", "bfloat16")))
        return case if case["batch"] * case["height"] * case["width"] * channels <= 30_000_000 else None
    case = dict(kind=kind, variant=rng.choice(tuple(_DEPTHS)), batch=_log_int(rng, 1, 128), image=32 * rng.randint(5, 12),
                dtype=rng.choice(("float16", "bfloat16")))
    return case if work(case)["flops"] <= work(dict(kind="model", variant="b", batch=128, image=224, dtype="float16"))["flops"] else None


def draw(rng):
    while True:
        case = _draw_one(rng)
        if case is not None:
            return case


def _pyramid(case):
    """[(H, W)] of the levels, a level's sides half of the one before (rounded up), and their pixels together."""
    h, w, levels = case["height"], case["width"], []
    for _ in range(_LEVELS):
        levels.append((h, w))
        h, w = (h + 1) // 2, (w + 1) // 2
    return levels, sum(a * b for a, b in levels)


def _row(groups):
    """Elements of a packed offset row: 27 of each group for a 3 x 3 kernel, padded to a multiple of 8."""
    return -(-groups * 27 // 8) * 8


def _offsets(case, shape, gen):
    # pixels: a bounded range, or the bell with tails that a trained layer's offsets have
    if case["offsets"] == "uniform":
        return (torch.rand(shape, generator=gen, device="cuda") * 2 - 1) * case["spread"]
    return torch.randn(shape, generator=gen, device="cuda") * case["spread"]


def _learnt_offsets(dcn):
    """Offsets and modulation as a trained layer has them (a fresh layer's are zero): sampling points spread by about a
    pixel, which the input moves by a fraction of one, and moderate weights that it changes a little."""
    used = dcn.group * 27
    with torch.no_grad():
        weight, bias = dcn.offset_mask.weight[:used].view(dcn.group, 27, -1), dcn.offset_mask.bias[:used].view(dcn.group, 27)
        weight[:, :18].normal_(std=0.3 * dcn.channels ** -0.5)
        bias[:, :18].normal_()
        weight[:, 18:].normal_(std=0.1 * dcn.channels ** -0.5)
        bias[:, 18:].normal_(std=0.3)


def _reference_points(case, batch, levels, gen):
    """(batch, queries, 2): the pixel centres of the pyramid for an encoder, free points for a decoder."""
    if case["queries"]:
        return torch.rand(batch, case["queries"], 2, generator=gen, device="cuda") * 0.9 + 0.05
    points = []
    for h, w in levels:
        y, x = torch.meshgrid((torch.arange(h, device="cuda") + 0.5) / h, (torch.arange(w, device="cuda") + 0.5) / w, indexing="ij")
        points.append(torch.stack((x, y), -1).reshape(-1, 2))
    return torch.cat(points).expand(batch, -1, -1)


def prepare(case, seed):
    torch.manual_seed(seed)            # the modules' own initialisation
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]

    def normal(*shape):
        return torch.randn(shape, generator=gen, device="cuda")

    if kind == "dcnv4":
        dtype = _DTYPES[case["dtype"]]
        b, h, w, g, d = (case[k] for k in ("batch", "height", "width", "groups", "group_width"))
        rows = torch.zeros(b, h, w, _row(g), device="cuda")
        rows[..., :g * 27] = torch.cat((_offsets(case, (b, h, w, g, 18), gen), normal(b, h, w, g, 9)), -1).flatten(-2)
        state = dict(value=normal(b, h, w, g * d).to(dtype), rows=rows.to(dtype), args=(3, 3, 1, 1, 1, 1, 1, 1, g, d, 1.0, 256, 0))
        if case["train"]:
            state["value"].requires_grad_()
            state["rows"].requires_grad_()
            state["grad"] = normal(b, h, w, g * d).to(dtype)
        return dict(state, kind=kind, train=case["train"])

    if kind in ("attention", "attention_layer"):
        levels, pixels = _pyramid(case)
        b = case["batch"]
        queries = case["queries"] or pixels
        shapes = torch.tensor(levels, dtype=torch.int64, device="cuda")
        starts = torch.tensor([sum(x * y for x, y in levels[:i]) for i in range(_LEVELS)], dtype=torch.int64, device="cuda")
        reference = _reference_points(case, b, levels, gen)
        if kind == "attention":
            dtype = _DTYPES[case["dtype"]]
            wh = shapes.flip(-1).float()[:, None]
            # a few pixels of each level around the query, as the learnt offsets of an encoder or decoder are
            locations = reference[:, :, None, None, None] + 3.0 * normal(b, queries, _HEADS, _LEVELS, _POINTS, 2) / wh
            packed = torch.cat((locations.flatten(-3), normal(b, queries, _HEADS, _LEVELS * _POINTS)), -1).to(dtype)
            state = dict(value=normal(b, pixels, _HEADS, _HEAD_WIDTH).to(dtype), packed=packed, shapes=shapes, starts=starts)
            if case["train"]:
                state["value"].requires_grad_()
                state["packed"].requires_grad_()
                state["grad"] = normal(b, queries, _HEADS * _HEAD_WIDTH).to(dtype)
            return dict(state, kind=kind, train=case["train"])
        width = _HEADS * _HEAD_WIDTH
        with torch.device("cuda"):
            layer = FlashDeformAttn(width, _LEVELS, _HEADS, _POINTS)
        torch.nn.init.normal_(layer.sampling_offsets.weight, std=width ** -0.5)
        torch.nn.init.normal_(layer.attention_weights.weight, std=width ** -0.5)
        reference = reference[:, :, None].expand(-1, -1, _LEVELS, -1)
        if case["boxes"]:
            size = torch.rand(reference.shape, generator=gen, device="cuda") * 0.3 + 0.02
            reference = torch.cat((reference, size), -1)
        # pictures of a batch differ in size: each is padded at the right up to the widest
        share = 1.0 - 0.25 * torch.arange(b, device="cuda") / b
        padding = torch.cat([(torch.arange(w, device="cuda")[None, None] >= share[:, None, None] * w).expand(b, h, w).flatten(1)
                             for h, w in levels], 1)
        return dict(kind=kind, layer=layer, query=normal(b, queries, width).requires_grad_(), reference=reference.contiguous(),
                    features=normal(b, pixels, width).requires_grad_(), shapes=shapes, starts=starts, padding=padding,
                    grad=normal(b, queries, width).to(_DTYPES.get(case["amp"], torch.float32)), amp=case["amp"])

    if kind == "block":
        b, h, w, c = (case[k] for k in ("batch", "height", "width", "channels"))
        post = case["post_norm"]
        with torch.device("cuda"):
            # the settings of the T (pre-norm) and of the S and B variants (post-norm, depthwise layer, layer scale)
            layer = InternImageLayer(c, case["groups"], post_norm=post, layer_scale=0.2 if post else None,
                                     offset_scale=0.5 if post else 1.0, dw_kernel_size=3 if post else None)
        _learnt_offsets(layer.dcn)
        # with post-norm the residual stream under autocast is single precision, else it has the autocast type
        dtype = torch.float32 if post else _DTYPES[case["amp"]]
        return dict(kind=kind, layer=layer, params=list(layer.parameters()), x=normal(b, h * w, c).to(dtype).requires_grad_(),
                    shape=(h, w), grad=normal(b, h * w, c).to(dtype), amp=_DTYPES[case["amp"]])

    dtype = _DTYPES[case["dtype"]]
    with torch.device("cuda"):
        model = flash_intern_image(case["variant"])
    for level in model.levels:
        for layer in level.blocks:
            _learnt_offsets(layer.dcn)
            if layer.layer_scale:
                layer.gamma1.data.fill_(0.2)
                layer.gamma2.data.fill_(0.2)
    return dict(kind=kind, model=model.to(dtype).eval(), images=normal(case["batch"], 3, case["image"], case["image"]).to(dtype))


def run(state):
    kind = state["kind"]
    if kind == "model":
        with torch.no_grad():
            return state["model"](state["images"])
    if kind == "block":
        with torch.autocast("cuda", dtype=state["amp"]):
            out = state["layer"](state["x"], state["shape"])
        return (out.detach(), *torch.autograd.grad(out, [state["x"], *state["params"]], state["grad"]))
    if kind == "attention_layer":
        with torch.autocast("cuda", dtype=torch.float16, enabled=state["amp"] != "none"):
            out = state["layer"](state["query"], state["reference"], state["features"], state["shapes"], state["starts"],
                                 state["padding"])
        wanted = [state["query"], state["features"], *state["layer"].parameters()]
        return (out.detach(), *torch.autograd.grad(out, wanted, state["grad"]))
    if kind == "attention":
        inputs = [state["value"], state["packed"]]
        call = lambda: FlashDeformAttnFunction.apply(inputs[0], state["shapes"], state["starts"], inputs[1], 64, _POINTS)
    else:
        inputs = [state["value"], state["rows"]]
        call = lambda: DCNv4Function.apply(*inputs, *state["args"])
    if not state["train"]:
        with torch.no_grad():
            return call()
    out = call()
    return (out.detach(), *torch.autograd.grad(out, inputs, state["grad"]))


def work(case):
    """Bytes: every tensor that goes in or comes out, once (of a training pass: the output, its gradient and the inputs'
    gradients too). Operations: products and additions of the matrix products, and 8 for each sampled channel."""
    kind = case["kind"]
    if kind == "dcnv4":
        size = 4 if case["dtype"] == "float32" else 2
        pixels = case["batch"] * case["height"] * case["width"]
        channels, row = case["groups"] * case["group_width"], _row(case["groups"])
        if case["train"]:        # value, rows, output; gradient of the output in, of value and rows out
            return {"bytes": size * pixels * (4 * channels + 2 * row), "flops": 3 * 72 * pixels * channels}
        return {"bytes": size * pixels * (2 * channels + row), "flops": 72 * pixels * channels}
    if kind in ("attention", "attention_layer"):
        pixels = case["batch"] * _pyramid(case)[1]
        queries = case["batch"] * case["queries"] or pixels
        width, points = _HEADS * _HEAD_WIDTH, _HEADS * _LEVELS * _POINTS
        sampling = 8 * queries * _LEVELS * _POINTS * width
        if kind == "attention":
            size = 4 if case["dtype"] == "float32" else 2
            if case["train"]:
                return {"bytes": size * (2 * pixels * width + 6 * queries * points + 2 * queries * width), "flops": 3 * sampling}
            return {"bytes": size * (pixels * width + 3 * queries * points + queries * width), "flops": sampling}
        weights = 2 * width * width + 3 * width * points
        products = 2 * pixels * width * width + 2 * queries * width * (width + 3 * points)
        ref = queries * _LEVELS * (4 if case["boxes"] else 2)
        return {"bytes": 4 * (2 * pixels * width + 4 * queries * width + ref + 2 * weights) + pixels,
                "flops": 3 * (products + sampling)}
    if kind == "block":
        tokens, c = case["batch"] * case["height"] * case["width"], case["channels"]
        weights = c * (10 * c + _row(case["groups"]))
        size = 4 if case["post_norm"] else 2
        return {"bytes": size * 4 * tokens * c + 8 * weights, "flops": 3 * tokens * (2 * weights + 72 * c)}
    b, side, c0 = case["batch"], case["image"] // 4, _CHANNELS[case["variant"]]
    flops = 2 * b * (4 * side * side * 27 * (c0 // 2) + side * side * 9 * (c0 // 2) * c0)
    params = 27 * (c0 // 2) + 9 * (c0 // 2) * c0
    for i, depth in enumerate(_DEPTHS[case["variant"]]):
        c, tokens = c0 << i, b * (side >> i) ** 2
        layer = c * (10 * c + _row(c // 16))
        flops += depth * tokens * (2 * layer + 72 * c)
        params += depth * layer
        if i < 3:
            flops += 2 * 18 * c * c * b * (side >> (i + 1)) ** 2
            params += 18 * c * c
    last = c0 * 8
    flops += 2 * b * ((side >> 3) ** 2 * last * last * 3 // 2 + last * 3 // 2 * 1000)
    params += last * last * 3 // 2 + last * 3 // 2 * 1000
    return {"bytes": 2 * (params + b * (3 * case["image"] ** 2 + 1000)), "flops": flops}


def tolerance(case):
    """What rounding gives: 32-bit sums in another order; one rounding of a result to 16 bits; and for layers and models a
    chain of 16-bit intermediates. In training such a chain rounds the sampling points too, and a gradient by a sampling
    point jumps where the point crosses a pixel: measured against single precision, up to 1.6e-2 for float16. The attention
    layer in single precision rounds its locations through fp16."""
    kind = case["kind"]
    if kind in ("dcnv4", "attention"):
        return {"float32": {"rel": 2e-5, "max": 2e-3}, "float16": {"rel": 2e-3}, "bfloat16": {"rel": 1e-2}}[case["dtype"]]
    if kind == "model":
        return {"rel": 3e-3 if case["dtype"] == "float16" else 1.5e-2}
    return {"rel": {"none": 2e-3, "float16": 2e-2, "bfloat16": 3e-2}[case["amp"]]}
