"""Depth ranks of more keys than one workgroup's LDS holds (sorted blocks,
merged segments, searches across segments) at the counts where a path begins or
ends, with ties, one key everywhere, sorted and reversed keys and NaN bits:
the stable order of numpy, for the Gaussian and the cubic binning."""
import numpy as np
import pytest
import torch

KINDS = ("random", "ties", "equal", "ascending", "descending", "special")


def _depths(kind, n):
    rng = np.random.default_rng(n)
    if kind == "random":
        return rng.standard_normal(n).astype(np.float32)
    if kind == "ties":
        return rng.integers(0, 5, n).astype(np.float32)
    if kind == "equal":
        return np.full(n, 0.7310586, np.float32)
    if kind == "ascending":
        return np.linspace(0, 1, n, dtype=np.float32)
    if kind == "descending":
        return np.linspace(1, 0, n, dtype=np.float32)
    return rng.choice(np.array([0.0, -0.0, np.nan, np.inf, -np.inf, 1e-40, 3.0], np.float32), n)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [8193, 16384, 16385, 20481, 24576, 65536, 100003, 262144, 262145])
@pytest.mark.parametrize("kind", KINDS)
def test_gaussian_depth_order(n, kind):
    from repo_amd import gaussian as G
    print(f"[ranks] {n} {kind}", flush=True)
    d = _depths(kind, n)
    xy = torch.rand((n, 2), device="cuda") * 60
    q = torch.tensor([1.0, 0.0, 1.0], device="cuda").repeat(n, 1)
    radii = torch.full((n,), 3, dtype=torch.int32, device="cuda")
    b = G.bin_gaussians(xy, q, radii, torch.from_numpy(d).cuda(), 64, 64, 16, 16)
    want = np.argsort(d.view(np.uint32), kind="stable")
    np.testing.assert_array_equal(b.order.cpu().numpy(), want)
    rects = b.tile_rects.cpu().numpy()[want]
    np.testing.assert_array_equal(b.rank_tile_ranges.cpu().numpy(), rects)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [16385, 30000, 262145])
def test_stroke_depth_order(n):
    """The cubic path (its blocks are ranked by the record launch); its key
    orders negative depths too (bits ^ ((bits >> 31) | 0x80000000))."""
    from repo_amd import splat
    print(f"[ranks] strokes {n}", flush=True)
    d = _depths("random", n)
    cub = torch.rand((n, 4, 2), device="cuda") * 2 - 1
    cub = cub[:, :1] + 0.02 * cub
    one = torch.ones(n, device="cuda")
    b = splat.bin_primitives(cub.contiguous(), torch.arange(n + 1, dtype=torch.int32, device="cuda"),
                             torch.rand((n, 3), device="cuda"), one, torch.from_numpy(d).cuda(),
                             None, one, one, 64, 80, 4, mode=splat.MODE_STROKE)
    np.testing.assert_array_equal(b.order.cpu().numpy(), np.argsort(d, kind="stable"))
