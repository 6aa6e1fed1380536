"""The window gathers of the DCNv4 operator at the edges of their tiles, against the oracle: every lanes-per-group and
groups-per-workgroup variant, images smaller than a tile, one pixel into the next tile and of a row, groups left over in the last
workgroup, points beyond the window and outside the image."""
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
