"""Filled chains with gaps between their segments, as an optimizer leaves them
(each segment's copy of a shared end point moves by itself): the raster sums
the crossings of the edges right of a wave per pixel row from their cull words.
Chains of fewer and more than 64, 256 and 384 edges, gaps below and above a pixel, long
spirals (winding numbers beyond a byte) and both fill rules, bit for bit
against the oracle, and the gradients."""
import math

import numpy as np
import pytest
import torch

from helpers import check_grads, hip_bin, oracle_forward, random_v_out
from oracle import oracle as O
from repo_amd import _native as N
from repo_amd import splat, synth

# Canvases of launches with eight waves on a 16 x 8 block, with four and with
# one (120, 600 and 1332 sub-blocks); the scenes grow with them.
CANVASES = {8: (150, 190), 4: (371, 393), 1: (561, 577)}


def _drifted(seed, drift, nseg, S, H, W, P=24):
    sc = synth.small_scene(seed, P=P, nseg=nseg, h=H, w=W, S=S, rmin=4.0, rmax=0.47 * H)
    g = torch.Generator("cpu").manual_seed(seed + 77)
    half = torch.tensor([W / 2.0, H / 2.0])
    sc.cubics_norm = sc.cubics_norm + drift * torch.randn(sc.cubics_norm.shape, generator=g) / half
    sc.fill_rules = (torch.arange(P) % 3 != 0).to(torch.int32)
    return sc


def _spiral(turns, H, W, S=4):
    """One chain of `turns` loops around the image centre (4 cubics a loop,
    shrinking), ending away from its start, above a drifted scene."""
    sc = _drifted(5, 0.02, 4, S, H, W, P=6)
    k = torch.arange(4 * turns + 1, dtype=torch.float32)
    th, r = k * (math.pi / 2), 0.4 * H - 10.0 * k / k[-1]
    p = torch.stack([W / 2 + r * th.cos(), H / 2 + r * th.sin()], 1)
    t = torch.stack([-th.sin(), th.cos()], 1) * (r * 0.5523).unsqueeze(1)
    cub = torch.stack([p[:-1], p[:-1] + t[:-1], p[1:] - t[1:], p[1:]], 1)
    half = torch.tensor([W / 2.0, H / 2.0])
    n0 = int(sc.seg_offsets[-1])
    sc.cubics_norm = torch.cat([sc.cubics_norm, cub / half - 1.0]).contiguous()
    sc.seg_offsets = torch.cat([sc.seg_offsets,
                                torch.tensor([n0 + cub.shape[0]], dtype=torch.int32)])
    one = torch.ones(1)
    sc.colors = torch.cat([sc.colors, torch.rand(1, 3)])
    sc.opacities = torch.cat([sc.opacities, 0.7 * one])
    sc.depths = torch.cat([sc.depths, 0.01 * one])
    sc.aa_widths = torch.cat([sc.aa_widths, one])
    sc.fill_rules = torch.cat([sc.fill_rules, torch.ones(1, dtype=torch.int32)])
    return sc


SCENES = {
    "tiny_gaps": lambda h, w: _drifted(0, 0.02, 4, 16, h, w),
    "pixel_gaps": lambda h, w: _drifted(1, 1.5, 4, 16, h, w),
    "exactly_64_edges": lambda h, w: _drifted(2, 0.3, 4, 17, h, w),
    "two_chunks": lambda h, w: _drifted(3, 0.3, 3, 24, h, w),
    "four_chunks": lambda h, w: _drifted(4, 0.3, 9, 24, h, w),
    "six_chunks": lambda h, w: _drifted(6, 0.3, 15, 24, h, w),
    "closed_three_chunks": lambda h, w: _drifted(7, 0.0, 7, 24, h, w),
    "256_edges": lambda h, w: _drifted(8, 0.05, 16, 17, h, w),
    "closed_384_edges": lambda h, w: _drifted(9, 0.0, 24, 17, h, w),
    "closed_seven_chunks": lambda h, w: _drifted(10, 0.0, 17, 24, h, w),
    "winding_beyond_a_byte": lambda h, w: _spiral(150, h, w),
}


def _bits(a):
    return np.ascontiguousarray(a).view(np.int32)


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(SCENES))
@pytest.mark.parametrize("waves,counted", [(8, False), (8, True), (4, False), (1, False)])
def test_far_edges_count_per_row(name, waves, counted):
    """(The counting instances always take one wave.)"""
    h, w = CANVASES[waves]
    for backward in (0, 1):
        assert N.lib().cs_raster_split_waves(splat.MODE_FILL, splat.sub_blocks(h, w),
                                             backward) == waves
    sc = SCENES[name](h, w)
    print(f"[far rows] {name} waves={waves} counted={counted}", flush=True)
    b, s = hip_bin(sc)
    bg = s.background.float().contiguous()
    counts = torch.zeros(5, dtype=torch.int64, device="cuda") if counted else None
    out, T, idx = splat.rasterize_forward(b, bg, eval_counts=counts)
    fw = oracle_forward(sc)
    np.testing.assert_array_equal(_bits(out.cpu().numpy()), _bits(fw["out"]))
    np.testing.assert_array_equal(_bits(T.cpu().numpy()), _bits(fw["final_T"]))
    np.testing.assert_array_equal(idx.cpu().numpy(), fw["final_idx"])
    v = random_v_out(sc.img_h, sc.img_w, seed=3)
    v_px, v_col, v_op, v_is2, _ = splat.rasterize_backward(b, bg, T, idx, v.cuda(),
                                                           eval_counts=counts)
    g = O.render_backward(fw, v.numpy())
    check_grads([("v_colors", v_col, g["v_colors"]), ("v_opacities", v_op, g["v_opacities"]),
                 ("v_inv_sigma2s", v_is2, g["v_inv_sigma2s"]),
                 ("v_cubics_px", v_px, g["v_cubics_px"])])
