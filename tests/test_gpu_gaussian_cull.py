"""The Gaussian raster's per-wave cull (an entry is left out when its ellipse
misses the wave's pixels) and its one- and two-pixel launches, against the
oracle, which evaluates every entry at every pixel: needles, discs and dots at
every offset from the pixel blocks, indefinite and non-finite conics, opacities
at the threshold."""
import numpy as np
import pytest
import torch

from helpers import grad_scale_tol
from oracle import oracle as O

# name: (n, H, W, block_x, block_y); two pixels per lane from 6144 waves of 128
# pixels on in the forward and 2048 in the backward (6240, 2080 and 8694 here).
CASES = {
    "one_pixel_16x8": (600, 120, 150, 16, 8),
    "odd_block_5x7": (300, 60, 70, 5, 7),
    "wide_block_128x2": (300, 50, 260, 128, 2),
    "one_wave_of_64": (300, 64, 96, 8, 8),
    "two_pixels_16x8": (400, 768, 1030, 16, 8),
    "two_pixels_backward_16x8": (400, 256, 1030, 16, 8),
    "two_pixels_24x16": (400, 736, 1500, 24, 16),
}


def _scene(name):
    n, H, W, bx, by = CASES[name]
    rng = np.random.default_rng(len(name))
    f = np.float32
    xy = np.stack([rng.uniform(-10, W + 10, n), rng.uniform(-10, H + 10, n)], 1).astype(f)
    th = rng.uniform(0, np.pi, n)
    s = np.exp(rng.uniform(np.log(0.3), np.log(40.0), (n, 2)))
    cs, sn = np.cos(th), np.sin(th)
    q = np.stack([(cs / s[:, 0]) ** 2 + (sn / s[:, 1]) ** 2,
                  sn * cs * (1 / s[:, 0] ** 2 - 1 / s[:, 1] ** 2),
                  (sn / s[:, 0]) ** 2 + (cs / s[:, 1]) ** 2], 1).astype(f)
    opac = rng.uniform(0.0, 1.0, n).astype(f)
    opac[::17] = f(1 / 255) * f(1.0001)
    opac[1::29] = 0.0
    q[2::31, 1] = 2.0 * np.sqrt(q[2::31, 0] * q[2::31, 2])   # indefinite
    q[3::41, 0] = -q[3::41, 0]
    q[4::97] = [np.inf, 0.0, 1.0]
    xy[5::89, 0] = np.nan
    # Centres on the blocks' sides and corners.
    xy[6::13] = np.round(xy[6::13] / [bx, by]) * [bx, by]
    radii = rng.integers(1, 60, n).astype(np.int32)
    dep = rng.uniform(0, 1, n).astype(f)
    ok = np.isfinite(xy).all(1) & np.isfinite(q).all(1)
    # Every entry in every tile its square reaches (odd ones in a few tiles).
    rx = np.where(ok, radii, 4)
    ids, tiles = [], []
    tbx, tby = -(-W // bx), -(-H // by)
    for g in np.argsort(dep, kind="stable"):
        cx, cy = (xy[g] if ok[g] else (W / 2, H / 2))
        x0, x1 = int(max(0, (cx - rx[g]) // bx)), int(min(tbx, (cx + rx[g]) // bx + 1))
        y0, y1 = int(max(0, (cy - rx[g]) // by)), int(min(tby, (cy + rx[g]) // by + 1))
        for ty in range(y0, y1):
            for tx in range(x0, x1):
                ids.append(g)
                tiles.append(ty * tbx + tx)
    ids, tiles = np.array(ids, np.int32), np.array(tiles)
    at = np.argsort(tiles, kind="stable")
    ids, tiles = ids[at], tiles[at]
    lo = np.searchsorted(tiles, np.arange(tbx * tby), "left")
    hi = np.searchsorted(tiles, np.arange(tbx * tby), "right")
    bins = np.stack([lo, hi], 1).astype(np.int32)
    return xy, q, rng.uniform(0, 1, (n, 3)).astype(f), opac, ids, bins


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
def test_cull_changes_nothing(name):
    from repo_amd import gaussian as G
    n, H, W, bx, by = CASES[name]
    print(f"[gs cull] {name}", flush=True)
    xy, q, c, o, ids, bins = _scene(name)
    bg = np.array([0.2, 0.4, 0.8], np.float32)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    rec = G.pack_records(dev(xy), dev(q), dev(c), dev(o))
    out, T, idx = G.rasterize_forward(dev(ids), dev(bins), rec, dev(bg), H, W, bx, by)
    r_out, r_T, r_idx = O.gs_raster_forward(ids, bins, xy, q, c, o, bg, H, W, bx, by)
    np.testing.assert_array_equal(idx.cpu().numpy(), r_idx)
    np.testing.assert_array_equal(T.cpu().numpy(), r_T)
    np.testing.assert_array_equal(out.cpu().numpy(), r_out)
    # Gradients over the finite records (the others' own are not finite).
    fine = np.isfinite(xy).all(1) & np.isfinite(q).all(1) & (q[:, 0] > 0)
    v = np.random.default_rng(3).standard_normal((H, W, 3)).astype(np.float32)
    contrib = torch.zeros((n, 3), device="cuda")
    got = G.rasterize_backward(dev(ids), dev(bins), rec, dev(bg), H, W, bx, by, T, idx, dev(v),
                               curve_contrib_rgb=contrib)
    plain = G.rasterize_backward(dev(ids), dev(bins), rec, dev(bg), H, W, bx, by, T, idx, dev(v))
    want = O.gs_raster_backward(ids, bins, xy, q, c, o, bg, H, W, bx, by, r_T, r_idx, v)
    for k in range(4):
        w = np.asarray(want[k])[fine]
        assert np.isfinite(w).all()   # (else nothing would be compared)
        for g in (got[k], plain[k]):
            ok, rel = grad_scale_tol(g.cpu().numpy()[fine], w, rtol=2e-4)
            assert ok, (name, k, rel)
    ok, rel = grad_scale_tol(contrib.cpu().numpy()[fine], np.asarray(want[4])[fine], rtol=2e-4)
    assert ok, rel
