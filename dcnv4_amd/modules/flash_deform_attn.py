"""``FlashDeformAttn`` layer: multi-scale deformable attention (Deformable DETR) on the fused sampling operator.

What the reference fixes and this module keeps (DCNv4_op/DCNv4/modules/flash_deform_attn.py:30-144): constructor
arguments, parameter names and creation order, the initial values (offset biases on a square ring around the
reference point, one direction per head, the k-th point k steps out; zero offset and attention weights; Xavier
projections), ``im2col_step = 64``, the forward signature and its arithmetic - including the passage of the sampling
locations through fp16 before they meet the attention logits.
"""
import math
import warnings

import torch
from torch import nn

from .. import ext
from ..functions import FlashDeformAttnFunction, FlashDeformAttnSplitFunction
from ..functions.flash_deform_attn_func import _interpreted


def _ring_directions(n_heads):
    """One unit-max-norm direction per head, evenly spaced in angle: (n_heads, 2) with max(|x|, |y|) = 1."""
    angle = torch.arange(n_heads, dtype=torch.float32) * (2.0 * math.pi / n_heads)
    xy = torch.stack((angle.cos(), angle.sin()), dim=-1)
    return xy / xy.abs().amax(dim=-1, keepdim=True)


class FlashDeformAttn(nn.Module):
    def __init__(self, d_model=256, n_levels=4, n_heads=8, n_points=4):
        super().__init__()
        head_dim, rest = divmod(d_model, n_heads)
        if rest:
            raise ValueError(f"d_model ({d_model}) is not a multiple of n_heads ({n_heads})")
        if head_dim & (head_dim - 1):
            warnings.warn(f"head width {head_dim} is not a power of two: the gfx950 kernels pad a head's lanes to the "
                          "next power of two")
        self.im2col_step = 64
        self.d_model, self.n_levels, self.n_heads, self.n_points = d_model, n_levels, n_heads, n_points

        points = n_heads * n_levels * n_points
        self.sampling_offsets = nn.Linear(d_model, 2 * points)
        self.attention_weights = nn.Linear(d_model, points)
        self.value_proj = nn.Linear(d_model, d_model)
        self.output_proj = nn.Linear(d_model, d_model)
        self._reset_parameters()

    def _reset_parameters(self):
        steps = torch.arange(1, self.n_points + 1, dtype=torch.float32)                       # point k sits k steps out
        ring = _ring_directions(self.n_heads)[:, None, None, :] * steps[None, None, :, None]  # (heads, 1, points, 2)
        ring = ring.expand(self.n_heads, self.n_levels, self.n_points, 2)
        with torch.no_grad():
            self.sampling_offsets.weight.zero_()
            self.sampling_offsets.bias.copy_(ring.reshape(-1))
            self.attention_weights.weight.zero_()
            self.attention_weights.bias.zero_()
        for proj in (self.value_proj, self.output_proj):
            nn.init.xavier_uniform_(proj.weight)
            nn.init.zeros_(proj.bias)

    def _sampling_locations(self, offsets, reference_points, spatial_shapes):
        """Normalised (x, y) of every sampling point: (N, Lq, heads, levels, points, 2)."""
        ref = reference_points[:, :, None, :, None, :]            # broadcast over heads and points
        kind = reference_points.shape[-1]
        if kind == 2:       # points: offsets are in pixels of each level
            wh = spatial_shapes.flip(-1)[None, None, None, :, None, :]
            return ref + offsets / wh
        if kind == 4:       # boxes (cx, cy, w, h): offsets are in units of half a box per n_points
            return ref[..., :2] + offsets / self.n_points * ref[..., 2:] * 0.5
        raise ValueError(f"reference_points must end in 2 (points) or 4 (boxes) coordinates, got {kind}")

    def forward(self, query, reference_points, input_flatten, input_spatial_shapes, input_level_start_index,
                input_padding_mask=None):
        """query (N, Lq, C); reference_points (N, Lq, n_levels, 2 or 4) in [0, 1]; input_flatten (N, sum H_l W_l, C);
        input_spatial_shapes (n_levels, 2) int64 rows (H_l, W_l); input_level_start_index (n_levels,) int64;
        input_padding_mask (N, sum H_l W_l) bool, True where the input is padding.  Returns (N, Lq, C)."""
        if query.is_cuda and not _interpreted():
            # one call where the kernels take the layer as it is, checks included (csrc/binding/attention.cpp)
            out = ext._native.attention_layer(self, query, reference_points, input_flatten, input_spatial_shapes,
                                              input_level_start_index, input_padding_mask)
            if out is not None:
                return out

        n, n_query, _ = query.shape
        n_in = input_flatten.shape[1]
        # the shapes cannot be read while a graph records them
        if not (query.is_cuda and torch.cuda.is_current_stream_capturing()):
            assert input_spatial_shapes.prod(-1).sum() == n_in, "the levels do not add up to the flattened input"

        value = self.value_proj(input_flatten)
        if input_padding_mask is not None:
            value = value.masked_fill(input_padding_mask.unsqueeze(-1), 0.0)
        value = value.view(n, n_in, self.n_heads, self.d_model // self.n_heads)

        offsets = self.sampling_offsets(query).view(n, n_query, self.n_heads, self.n_levels, self.n_points, 2)
        logits = self.attention_weights(query).view(n, n_query, self.n_heads, self.n_levels * self.n_points)
        locations = self._sampling_locations(offsets, reference_points, input_spatial_shapes)

        # One row per (query, head): 2 L K locations, rounded through fp16 as in the reference (:132), and the L K
        # attention logits.  The operator takes the two tensors as they are and rounds while it stages them; dtype
        # mixes it does not take are packed with torch first, as the reference does.
        locations = locations.flatten(-3)
        if logits.dtype == value.dtype and locations.dtype in (torch.float32, value.dtype):
            sampled = FlashDeformAttnSplitFunction.apply(value, input_spatial_shapes, input_level_start_index,
                                                         locations.contiguous(), logits.contiguous(), self.im2col_step,
                                                         self.n_points)
        else:
            packed = torch.cat((locations.half(), logits), dim=-1)
            sampled = FlashDeformAttnFunction.apply(value, input_spatial_shapes, input_level_start_index, packed,
                                                    self.im2col_step, self.n_points)
        return self.output_proj(sampled)


ext._native.register_modules(FlashDeformAttn)
