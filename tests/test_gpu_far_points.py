"""DCNv4 backward where some sampling points lie far from their pixel: the tiles of the input gradient are visited by the pixels
around them, and the points that land in one from farther away are listed (images of several tiles each way).  Against the oracle:
tails of every length, a few outliers, a region where most points are far, and one that collects more of them than a list holds."""
import pytest
import torch

from tests import cabi
from tests.test_gpu_parity import GRAD_TOL, _dcn_inputs, _oracle_args

pytestmark = pytest.mark.gpu

GEOM = (3, 3, 1, 1, 1, 1, 1, 1)
# batch, height, width, groups, group width: many tiles, a ragged one, one row of them; two chunks of groups; wide groups
SHAPES = [(2, 109, 131, 3, 16), (1, 130, 21, 2, 32), (1, 47, 64, 5, 64)]


def _offsets(kind, rows, groups):
    """rows [B, H, W, groups * 27 ..]: the offsets replaced by those of the kind."""
    b, h, w, _ = rows.shape
    gen = torch.Generator().manual_seed(h)
    off = torch.randn(b, h, w, groups, 9, 2, generator=gen)
    if kind == "bell":
        off *= 2.5
    elif kind == "outliers":                     # some of them out of the image
        off[torch.rand(off.shape[:-1], generator=gen) < 0.003] *= 30.
    elif kind == "region":
        off[:, : h // 3] = (torch.rand(off[:, : h // 3].shape, generator=gen) * 2 - 1) * 20.
    else:                                        # one point of every pixel goes to the middle of the image
        centre = torch.stack(torch.broadcast_tensors(torch.arange(w)[None, :] - w / 2, torch.arange(h)[:, None] - h / 2), -1)
        off[..., 4, :] = 4. * off[..., 4, :] - centre[None, :, :, None]
    rows[..., :groups * 27].view(b, h, w, groups, 27)[..., :18] = off.flatten(-2).to(rows.dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("kind", ["bell", "outliers", "region", "magnet"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(str(v) for v in s))
def test_backward_with_far_points_matches_oracle(oracle, shape, kind, dtype):
    v, om, go, (geom, G, D, scale, rc) = _dcn_inputs((*shape, GEOM, 0, 1.0, 1.0), dtype, seed=7)
    _offsets(kind, om, G)
    args = _oracle_args(geom, G, D, scale, rc)
    wgv, wgom = oracle.dcnv4_backward(cabi.f64(v), cabi.f64(om), cabi.f64(go), *args, coord_f32=True)
    print(f"far points {shape} {kind} {dtype}", flush=True)
    for _ in range(2):                           # the second call finds the lists that the first one left in a reused buffer
        state = []
        gv, gom = cabi.dcnv4_backward(v.cuda(), om.cuda(), go.cuda(), geom, G, D, scale, rc, state=state)
        torch.cuda.synchronize()
        # GradState: whether lists were written, from word 8 on visits widened for points that no list holds.  The kernel that lists takes
        # groups of up to 128 bytes; of a region's points most leave the narrow image
        words = state[0][:64].tolist()
        assert words[0] == (D * v.element_size() <= 128)
        assert not words[0] or any(words[8:]) == (kind == "magnet" or kind == "region" and shape[2] > 40)
        cabi.assert_close(gv, wgv, *GRAD_TOL[dtype], what="grad_value")
        cabi.assert_close(gom, wgom, *GRAD_TOL[dtype], what="grad_offset_mask")


def test_backward_into_the_memory_of_its_input(oracle):
    """grad_value is scratch memory for the lists only where no input lies: the result may replace the value."""
    from dcnv4_amd import _lib
    v, om, go, (geom, G, D, scale, rc) = _dcn_inputs((2, 109, 131, 3, 16, GEOM, 0, 1.0, 1.0), torch.float16, seed=7)
    _offsets("bell", om, G)
    vd, omd, god = v.cuda(), om.cuda(), go.cuda()
    want, want_om = cabi.dcnv4_backward(vd, omd, god, geom, G, D, scale, rc)
    L, gom, ws = _lib.load(), torch.empty_like(omd), torch.empty(256, dtype=torch.uint8, device="cuda")
    _lib.check(L.dcnv4_gfx950_backward(vd.data_ptr(), omd.data_ptr(), god.data_ptr(), vd.data_ptr(), gom.data_ptr(), ws.data_ptr(), 256,
                                       _lib.DTYPE_F16, 2, 109, 131, G, D, *geom, scale, 256, rc, om.shape[-1], 0, 0, 0, cabi._stream()))
    torch.cuda.synchronize()
    assert ws[:4].view(torch.int32).item() == 0 and torch.equal(gom, want_om)
    cabi.assert_close(vd, cabi.f64(want), *GRAD_TOL[torch.float16], what="grad_value")
