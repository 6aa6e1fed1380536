"""The window gathers of the DCNv4 operator at the edges of their tiles, against the oracle: every lanes-per-group and
units-per-workgroup variant (which of them a shape takes follows from the bytes of a group, one lane for 32, and from the pixels:
two units a workgroup up to 64, four up to 32), images smaller than a tile, one pixel into the next tile and of a row, groups left
over in the last workgroup, points beyond the window and outside the image, offsets that are no numbers."""
import pytest
import torch

from tests import cabi
from tests.test_gpu_parity import FWD_TOL, GRAD_TOL, _dcn_inputs, _oracle_args

pytestmark = pytest.mark.gpu

# batch, height, width, groups, group width, reach of the window, spread of the offsets
SHAPES = [(3, 5, 3, 3, 16, 2, 3.0), (2, 17, 33, 3, 16, 5, 6.0), (1, 1, 40, 2, 32, 0, 2.0), (2, 15, 18, 3, 32, 4, 8.0),
          (1, 33, 2, 5, 32, 12, 20.0), (1, 9, 17, 3, 64, 4, 5.0)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(str(v) for v in s[:5]))
def test_window_gathers_match_oracle(oracle, shape, dtype):
    from dcnv4_amd import ext
    b, h, w, groups, width, reach, spread = shape
    case = (b, h, w, groups, width, (3, 3, 1, 1, 1, 1, 1, 1), 0, 1.0, spread)
    v, om, go, (geom, G, D, scale, rc) = _dcn_inputs(case, dtype, seed=h)
    args = _oracle_args(geom, G, D, scale, rc)
    want = oracle.dcnv4_forward(cabi.f64(v), cabi.f64(om), *args, coord_f32=True)
    wgv, wgom = oracle.dcnv4_backward(cabi.f64(v), cabi.f64(om), cabi.f64(go), *args, coord_f32=True)
    with ext.launch_options(reach=reach, dual="off"):      # a reach of one's own: small calls use the window too
        out = cabi.dcnv4_forward(v.cuda(), om.cuda(), geom, G, D, scale, rc)
        gv, gom = cabi.dcnv4_backward(v.cuda(), om.cuda(), go.cuda(), geom, G, D, scale, rc)
    torch.cuda.synchronize()
    cabi.assert_close(out, want, *FWD_TOL[dtype], what="output")
    cabi.assert_close(gv, wgv, *GRAD_TOL[dtype], what="grad_value")
    cabi.assert_close(gom, wgom, *GRAD_TOL[dtype], what="grad_offset_mask")
    assert (gom[..., G * 27:] == 0).all(), "padded tail of grad_offset_mask must be exactly zero"


# lanes and units that the shapes above leave out in 16 bits: (1, 2), two groups of 32 bytes on 33 to 64 pixels (the last stage of a
# model at 224 pixels), and (2, 4), two groups of 64 bytes on up to 32; an odd number of groups each, and one group alone
SMALL = [(3, 7, 7, 5, 16, 5, 3.0), (2, 1, 33, 1, 16, 0, 2.0), (2, 8, 8, 2, 16, 12, 20.0), (2, 5, 6, 3, 32, 2, 4.0), (1, 32, 1, 1, 32, 5, 3.0)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("shape", SMALL, ids=lambda s: "x".join(str(v) for v in s[:5]))
def test_window_gathers_of_small_images_match_oracle(oracle, shape, dtype):
    test_window_gathers_match_oracle(oracle, shape, dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("width", [16, 32, 64])
def test_window_gathers_drop_offsets_that_are_no_numbers(width, dtype):
    """Such a point is outside the image: it adds nothing, and its gradients are zero, as for one far outside."""
    from dcnv4_amd import ext
    b, h, w, groups = 2, 9, 13, 3
    case = (b, h, w, groups, width, (3, 3, 1, 1, 1, 1, 1, 1), 0, 1.0, 2.0)
    v, om, go, (geom, G, D, scale, rc) = _dcn_inputs(case, dtype, seed=width)
    results = []
    for values in ((float("nan"), float("inf"), float("-inf")), (1000.0, 1000.0, -1000.0)):
        rows = om.clone()
        for i, value in enumerate(values):
            rows[..., 2 * i] = value
            rows[:, 3, :, 27 + 2 * i + 7] = value
        with ext.launch_options(reach=4, dual="off"):
            out = cabi.dcnv4_forward(v.cuda(), rows.cuda(), geom, G, D, scale, rc)
            gv, gom = cabi.dcnv4_backward(v.cuda(), rows.cuda(), go.cuda(), geom, G, D, scale, rc)
        results.append((out, gv, gom))
    for got, want in zip(*results):
        assert torch.isfinite(got).all()
        cabi.assert_close(got, cabi.f64(want), *GRAD_TOL[dtype], what="against points far outside")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("reach", [4, 0], ids=["window", "beyond"])
@pytest.mark.parametrize("width", [16, 32, 64])
def test_window_gathers_carry_infinite_modulations(oracle, width, reach, dtype):
    """An infinite modulation times corners of one sign is infinite, not NaN, whether the window serves the point or memory (reach 0,
    for a part of the points).  Pixels whose points all lie inside the image, between its pixels: no corner has the weight zero."""
    from dcnv4_amd import ext
    b, h, w, groups = 2, 11, 13, 3
    case = (b, h, w, groups, width, (3, 3, 1, 1, 1, 1, 1, 1), 0, 1.0, 2.0)
    v, om, _, (geom, G, D, scale, rc) = _dcn_inputs(case, dtype, seed=width)
    gen = torch.Generator().manual_seed(width)
    v = v.abs() + 0.5
    rows = om[..., :groups * 27].view(b, h, w, groups, 27)
    rows[..., :18] = ((torch.rand(rows[..., :18].shape, generator=gen) * 0.6 + 0.2) * torch.randn(rows[..., :18].shape, generator=gen).sign()).to(dtype)
    rows[..., 18:] = (torch.rand(rows[..., 18:].shape, generator=gen) + 0.1).to(dtype)
    number = torch.arange(b * h * w * groups).view(b, h, w, groups) % 10
    for tap in range(9):                          # one in ten of every tap, of either sign
        rows[..., 18 + tap][number == tap] = float("inf") if tap % 2 else float("-inf")
    want = oracle.dcnv4_forward(cabi.f64(v), cabi.f64(om), *_oracle_args(geom, G, D, scale, rc), coord_f32=True)
    with ext.launch_options(reach=reach, dual="off"):
        out = cabi.dcnv4_forward(v.cuda(), om.cuda(), geom, G, D, scale, rc)
    got, want = cabi.f64(out)[:, 2:-2, 2:-2], want[:, 2:-2, 2:-2]
    infinite = abs(want) == float("inf")
    assert infinite.any() and not infinite.all() and (got[infinite] == want[infinite]).all()
    cabi.assert_close(got[~infinite], want[~infinite], *FWD_TOL[dtype], what="the others")


@pytest.mark.parametrize("reach", [4, 0], ids=["window", "beyond"])
@pytest.mark.parametrize("width,dtype", [(16, torch.float32), (32, torch.float32), (16, torch.float16), (32, torch.float16), (64, torch.float16),
                                         (16, torch.bfloat16), (32, torch.bfloat16), (64, torch.bfloat16)])
def test_gradient_of_the_modulation_sums_neighbouring_words_apart(width, reach, dtype):
    """A corner's product with grad_out is two sums, of every other 4-byte word: words of 2^25, 1, -2^25, 1 give the number of ones,
    which a single sum loses next to 2^25.  Points on pixels, where the gradient of a modulation is one corner's product."""
    from dcnv4_amd import ext
    b, h, w, groups = 2, 9, 13, 3
    case = (b, h, w, groups, width, (3, 3, 1, 1, 1, 1, 1, 1), 0, 1.0, 0.0)
    v, om, go, (geom, G, D, scale, rc) = _dcn_inputs(case, dtype, seed=width)
    om.zero_()
    word = 1 if dtype == torch.float32 else 2      # channels
    for t, words in ((v, (2.0 ** 13, 1.0, -2.0 ** 13, 1.0)), (go, (2.0 ** 12, 1.0, 2.0 ** 12, 1.0))):
        pattern = torch.zeros(4, word)
        pattern[:, 0] = torch.tensor(words)
        t.copy_(pattern.flatten().repeat(t.numel() // (4 * word)).view(t.shape).to(dtype))
    with ext.launch_options(reach=reach, dual="off"):
        _, gom = cabi.dcnv4_backward(v.cuda(), om.cuda(), go.cuda(), geom, G, D, scale, rc)
    rows = gom[:, 1:-1, 1:-1, :groups * 27].reshape(b, h - 2, w - 2, groups, 27).cpu().float()
    assert (rows[..., 18:] == width // word // 2).all(), rows[..., 18:].unique()
    assert (rows[..., :18] == 0).all()      # all corners alike


def test_rows_of_offsets_that_lie_gigabytes_apart():
    """Eight rows of 16393 pixels whose offset rows have 4096 elements are 2.1 GB, more than an int holds: the last column of tiles is one
    pixel wide, so that a lane of grad_offset_mask's stores goes on eight rows further down."""
    h, w = 10, 16393
    gen = torch.Generator(device="cuda").manual_seed(0)
    v, go = (torch.randn(1, h, w, 16, generator=gen, device="cuda") for _ in range(2))
    packed = torch.randn(1, h, w, 32, generator=gen, device="cuda")
    wide = torch.zeros(1, h, w, 4096, device="cuda")
    wide[..., :27] = packed[..., :27]
    geom = (3, 3, 1, 1, 1, 1, 1, 1)
    _, want = cabi.dcnv4_backward(v, packed, go, geom, 1, 16, 1.0, 0)
    _, got = cabi.dcnv4_backward(v, wide, go, geom, 1, 16, 1.0, 0)
    assert torch.equal(got[..., :27], want[..., :27]) and not got[..., 27:].any()
