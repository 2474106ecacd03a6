"""Raster launches over small images, which put several waves on each 16 x 8
block of pixels: image, T and final index bit for bit against the one-wave
launch (the counting instance) at the sizes where the wave count changes, with
lists longer than a chunk, pixels that stop early and log pools that run full;
gradients and contribution outputs against the oracle."""
import numpy as np
import pytest
import torch

from helpers import check_grads, grad_scale_tol, hip_bin, oracle_forward, random_v_out
from oracle import oracle as O
from repo_amd import _native as N
from repo_amd import splat, synth


def _waves(mode, nsub, backward=0):
    return int(N.lib().cs_raster_split_waves(mode, nsub, backward))


@pytest.mark.parametrize("mode", [splat.MODE_FILL, splat.MODE_STROKE])
@pytest.mark.parametrize("backward", [0, 1])
def test_the_wave_count_falls_with_the_image(mode, backward):
    assert _waves(mode, 0, backward) == 0 and _waves(2, 5, backward) == 0
    counts = [_waves(mode, n, backward) for n in range(1, 4000)]
    assert counts[0] == 8 and counts == sorted(counts, reverse=True)
    assert _waves(mode, 1 << 20, backward) == 1


@pytest.mark.parametrize("mode,last", [(splat.MODE_FILL, 1152), (splat.MODE_STROKE, 2048)])
def test_log_pool_holds_a_block_for_each_wave_of_the_launch(mode, last):
    """The pool's size follows the launch's own wave count: past the last size
    that is split, one wave per 16 x 8 block."""
    assert _waves(mode, last) == 4 and _waves(mode, last + 1) == 1
    for nsub in (1, 512, 513, last, last + 1, 2305):
        _, size = splat.log_layout(("no such scene",), 1000, mode, nsub)
        regions = 16 * 2 * 1000 * splat.LOG_FIRST_UNITS_PER_ENTRY
        blocks = 2 * nsub * _waves(mode, nsub) * N.RASTER_LOG_BLOCK_BYTES
        assert 0 <= size - (16 + regions + regions // 4 + blocks + (1 << 20)) < 256


# name: (H, W, paths, stroke), by the sub-blocks where a wave count changes
# (forward 512, 1152 and 2048, backward 256, 1024 and 1408) and just past them.
SIZES = {
    "one_block": (9, 13, 150, False),
    "ragged": (75, 100, 300, False),
    "fill_512": (256, 512, 60, False),
    "fill_513": (144, 912, 60, False),
    "fill_1152": (384, 768, 60, False),
    "stroke_ragged": (75, 100, 400, True),
    "stroke_2048": (512, 1024, 80, True),
    "fill_256": (256, 256, 60, False),
    "fill_260": (208, 320, 60, False),
    "fill_1024": (512, 512, 80, False),
    "fill_1025": (400, 656, 80, False),
    "stroke_256": (256, 256, 60, True),
    "stroke_260": (208, 320, 60, True),
    "stroke_1408": (512, 704, 90, True),
    "stroke_1410": (480, 752, 90, True),
}
FORWARD = ("one_block", "ragged", "fill_512", "fill_513", "fill_1152", "stroke_ragged",
           "stroke_2048")
BACKWARD = ("one_block", "ragged", "stroke_ragged", "fill_513", "fill_256", "fill_260",
            "fill_1024", "fill_1025", "stroke_256", "stroke_260", "stroke_1408", "stroke_1410")


def _scene(name):
    h, w, P, stroke = SIZES[name]
    return synth.small_scene(len(name), P=P, nseg=4, h=h, w=w, S=12, stroke=stroke,
                             rmin=2.0, rmax=0.45 * min(h, w))


def _bits(a):
    return np.ascontiguousarray(a.cpu().numpy()).view(np.int32)


@pytest.mark.gpu
@pytest.mark.parametrize("name", FORWARD)
@pytest.mark.parametrize("flatten", ["bernstein", "de_casteljau"])
def test_split_equals_one_wave(name, flatten):
    sc = _scene(name)
    print(f"[split] {name} {flatten}", flush=True)
    b, s = hip_bin(sc, flatten_method=flatten)
    bg = s.background.float().contiguous()
    out, T, idx = splat.rasterize_forward(b, bg)
    ref = splat.rasterize_forward(b, bg, eval_counts=torch.zeros(5, dtype=torch.int64,
                                                                 device="cuda"))
    for got, want in zip((out, T, idx), ref):
        np.testing.assert_array_equal(_bits(got), _bits(want))
    nolog = splat.rasterize_forward(b, bg, log=False)
    for got, want in zip(nolog, ref):
        np.testing.assert_array_equal(_bits(got), _bits(want))


@pytest.mark.gpu
@pytest.mark.parametrize("name", BACKWARD)
@pytest.mark.parametrize("pool", [None, 1 << 14])
def test_split_backward(name, pool):
    """Gradients and contribution outputs, with a full log and with one whose
    pool runs full (missing entries are recomputed)."""
    sc = _scene(name)
    print(f"[split backward] {name} pool={pool}", flush=True)
    b, s = hip_bin(sc)
    bg = s.background.float().contiguous()
    out, T, idx = splat.rasterize_forward(b, bg, log_pool_bytes_override=pool)
    fw = oracle_forward(sc)
    v = random_v_out(sc.img_h, sc.img_w, seed=1)
    rgb = torch.zeros((b.nprim, 3), device="cuda")
    isect = torch.zeros((b.num_intersects,), device="cuda")
    v_px, v_col, v_op, v_is2, v_sw = splat.rasterize_backward(
        b, bg, T, idx, v.cuda(), curve_contrib_rgb=rgb, curve_isect_contrib=isect)
    g = O.render_backward(fw, v.numpy())
    checks = [("v_colors", v_col, g["v_colors"]), ("v_opacities", v_op, g["v_opacities"]),
              ("v_inv_sigma2s", v_is2, g["v_inv_sigma2s"]),
              ("v_cubics_px", v_px, g["v_cubics_px"])]
    if v_sw is not None:
        checks.append(("v_stroke_widths", v_sw, g["v_stroke_widths"]))
    check_grads(checks)
    # Contributions: every composited term once (sum over the entries equals
    # the sum over the primitives, and the image minus its background).
    total = float(isect.double().sum())
    assert abs(total - float(rgb.double().sum())) <= 1e-5 * abs(total)
    shown = float((out.double() - T.double().unsqueeze(2) * bg.double()).sum())
    assert abs(total - shown) <= 1e-5 * abs(shown)
    ok, err = grad_scale_tol(rgb.sum(0).cpu().numpy(),
                             (out - T.unsqueeze(2) * bg).double().sum((0, 1)).cpu().numpy(),
                             rtol=1e-5)
    assert ok, err
