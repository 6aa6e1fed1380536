"""grad_value of flash deformable attention by tiles: where the walk over tiles and their points turns a corner, against the oracle."""
import numpy as np
import pytest
import torch

from dcnv4_amd import ext
from tests import cabi
from tests.inputs import make_fda_inputs

pytestmark = pytest.mark.gpu

# B, levels, G, D, K, Q
CASES = {
    # 137 chunks of points: the words of a tile come in three groups; one level, cut finer because a tile holds thousands of points
    "groups_of_chunks": (1, [(16, 16)], 1, 8, 4, 140000),
    # tiles handed out as workgroups come free, pairs by die: levels of 1, 5 and many tiles, one of a single cell
    "handed_out": (2, [(70, 90), (9, 7), (1, 1), (12, 12)], 8, 32, 4, 3000),
    # ... two windows of channels, whose launches take turns with the counters, and a third of them
    "windows_take_turns": (1, [(30, 40), (4, 4)], 8, 72, 4, 1500),
    # pairs that the dies do not share evenly, points that are no power of two, a part of a block and of a step at every list's end
    "odd_pairs": (1, [(33, 17), (5, 3)], 3, 16, 6, 1111),
    # hardly a point to a tile: most steps are empty
    "empty_tiles": (1, [(100, 120), (50, 60)], 8, 32, 4, 9),
}


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16], ids=["fp32", "fp16"])
@pytest.mark.parametrize("name", list(CASES))
def test_grad_value_by_tiles(oracle, name, dtype):
    B, levels, G, D, K, Q = CASES[name]
    print(f"case {name} dtype {dtype}", flush=True)
    v, shp, st, sla, go = make_fda_inputs(B, levels, G, D, K, Q, seed=len(name), dtype=dtype, loc_lo=-0.05, loc_hi=1.05)
    args = (cabi.f64(v), shp.numpy(), st.numpy(), cabi.f64(sla))
    want, _ = oracle.flash_deform_attn_backward(*args, cabi.f64(go), K, coord_f32=True)
    sizes, _ = oracle.flash_deform_attn_backward(*args, np.abs(cabi.f64(go)), K, coord_f32=True)      # of a sum's terms: all weights are positive
    with ext.launch_options(scatter="tiled"):
        got = [cabi.fda_backward(v.cuda(), shp.cuda(), st.cuda(), sla.cuda(), go.cuda(), K)[0] for _ in range(2)]
    torch.cuda.synchronize()
    # a weight is right to a few units of fp32 (16 for the exponential's argument), an n-term sum to n of them, and a cell has about
    # 4 * Q * K / cells terms; the result is rounded to the type
    terms = 4 * 4 * Q * K / min(h * w for h, w in levels)
    bound = sizes * (16 + terms) * 2.0 ** -24 + (np.abs(want) * 2.0 ** -11 + 2.0 ** -24 if dtype == torch.float16 else 1e-30)
    for g in got:
        assert (np.abs(cabi.f64(g) - want) <= bound).all(), float((np.abs(cabi.f64(g) - want) / bound).max())


# The same turns with sides that are powers of two, for data whose sums are exact: one lost or doubled point of one cell shows.
# B, levels, G, D, K, Q, then which levels are cut finer and whether tiles are handed out (fda_grad_value_kernel's `shared`)
EXACT = {
    "groups_of_chunks": (1, [(16, 16)], 1, 8, 4, 140000, [True], False),
    "groups_handed_out": (1, [(16, 16)], 8, 8, 4, 140000, [True], True),
    "handed_out": (1, [(64, 128), (16, 8), (1, 1), (16, 16)], 8, 32, 4, 12000, [False, True, False, True], True),
    "windows_take_turns": (1, [(32, 64), (16, 16)], 8, 72, 4, 4000, [False, True], True),
    "odd_pairs": (1, [(32, 16), (4, 2)], 3, 16, 6, 1111, [False, False], False),
    "empty_tiles": (1, [(128, 128), (64, 64)], 8, 32, 4, 9, [False, False], False),
}


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16], ids=["fp32", "fp16"])
@pytest.mark.parametrize("name", list(EXACT))
def test_grad_value_by_tiles_has_every_point_once(oracle, name, dtype):
    """Positions in quarters of a pixel, eight or sixteen equal probabilities a query, gradients of 1 and -1: every term is a multiple of
    2^-8 and every sum exact in fp32, so that the result is the oracle's, rounded once."""
    B, levels, G, D, K, Q, finer, handed_out = EXACT[name]
    print(f"case {name} dtype {dtype}", flush=True)
    tiles = [ext._native.attention_tile(h, w, Q * K, len(levels) * B * G, dtype.itemsize) for h, w in levels]
    assert [t != ext._native.attention_tile(h, w, 1, 1, dtype.itemsize) for t, (h, w) in zip(tiles, levels)] == finer
    assert (B * G % 8 == 0 and Q * K * len(levels) >= 256 * sum(-(-h // th) * -(-w // tw) for (h, w), (th, tw) in zip(levels, tiles))) == handed_out
    g = torch.Generator().manual_seed(len(name))
    v, shp, st, sla, go = make_fda_inputs(B, levels, G, D, K, Q, seed=1, dtype=torch.float32)
    rows = sla[..., :len(levels) * K * 2].view(B, Q, G, len(levels), K, 2)
    for level, (h, w) in enumerate(levels):
        for axis, side in ((0, w), (1, h)):      # from a pixel outside to the last one
            quarters = torch.randint(-3, 4 * side, (B, Q, G, K), generator=g)
            rows[..., level, :, axis] = (quarters / 4 + 0.5) / side
    logits = sla[..., len(levels) * K * 2:]
    logits.zero_()
    points = len(levels) * K
    equal = 1 << (points.bit_length() - 1)
    logits.scatter_(-1, torch.rand(logits.shape, generator=g).argsort(-1)[..., equal:], -1000.0)      # the others have none
    go.copy_(torch.randint(0, 2, go.shape, generator=g) * 2 - 1)
    v, sla, go = v.to(dtype), sla.to(dtype), go.to(dtype)
    want, _ = oracle.flash_deform_attn_backward(cabi.f64(v), shp.numpy(), st.numpy(), cabi.f64(sla), cabi.f64(go), K, coord_f32=True)
    assert (want * 256 == np.rint(want * 256)).all() and np.abs(want).max() * 256 < 2 ** 24 and want.any()
    want = torch.from_numpy(want).to(dtype)
    with ext.launch_options(scatter="tiled"):
        for _ in range(2):
            got = cabi.fda_backward(v.cuda(), shp.cuda(), st.cuda(), sla.cuda(), go.cuda(), K)[0].cpu()
            assert torch.equal(got, want), (int((got != want).sum()), float((got - want).abs().max()))


# fp32 tensors with fewer points than a third of the pixels take the atomic scatter by themselves: on either side of where, both ways
# against each other
@pytest.mark.parametrize("batch,queries", [(2, 28), (2, 29), (2, 280), (2, 320), (6, 100), (6, 120)])
def test_few_points_choose_a_way(batch, queries):
    v, shp, st, sla, go = (t.cuda() for t in make_fda_inputs(batch, [(30, 34), (15, 17), (8, 9), (4, 5)], 8, 32, 4, queries, seed=3, dtype=torch.float32))
    assert ext._native.attention_backward_tiled(v, 4, queries, 4) == (3 * 16 * queries >= v.shape[1]) == (queries > 28)
    auto, rows = cabi.fda_backward(v, shp, st, sla, go, 4)
    sizes, _ = cabi.fda_backward(v, shp, st, sla, go.abs(), 4)
    for scatter in ("tiled", "atomic"):
        with ext.launch_options(scatter=scatter):
            one, one_rows = cabi.fda_backward(v, shp, st, sla, go, 4)
        # the same terms in another order, at most 4 * queries * 4 of them
        assert ((one - auto).abs() <= sizes * (2 * 16 * queries * 2.0 ** -24) + 1e-30).all(), scatter
        torch.testing.assert_close(one_rows, rows, rtol=1e-4, atol=1e-5)


def test_many_points_on_few_pixels_go_by_tiles_however_little_work_they_are():
    """Atomics of one address wait for each other: one head of 8 channels, 6875 queries on 4 x 4 pixels, 417 us against 73."""
    tiled = lambda pixels, heads, channels, levels, queries, dtype=torch.float32: ext._native.attention_backward_tiled(
        torch.empty(1, pixels, heads, channels, dtype=dtype, device="meta"), levels, queries, 4)
    assert tiled(16, 1, 8, 1, 6875) and tiled(16, 8, 32, 1, 214) and tiled(1600, 1, 8, 4, 1720) and tiled(80, 1, 8, 2, 3437)
    assert tiled(20197, 8, 32, 4, 421) and not tiled(20197, 8, 32, 4, 420) and tiled(20197, 8, 32, 4, 300, torch.float16)
    with ext.launch_options(scatter="tiled"):
        assert tiled(20197, 8, 32, 4, 300)
    with ext.launch_options(scatter="atomic"):
        assert not tiled(16, 1, 8, 1, 6875)
