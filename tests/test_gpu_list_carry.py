"""Tile lists of slabs with several chunks of 1024 ranks: hits held back over
chunks and dealt when another chunk might not fit (few hits a chunk, all 1024
of them, and both in turn), against the oracle's lists."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from repo_amd import gaussian as G

# 512 rows of tiles: at most two slabs, of up to nine chunks.
H, W, BX, BY = 512, 64, 16, 1


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n", [(k, n) for n in (1024, 2049, 5000)
                                    for k in ("few", "all", "turns")]
                         + [("few", 17000), ("turns", 17000)])
def test_lists_over_chunks(kind, n):
    print(f"[list carry] {kind} {n}", flush=True)
    rng = np.random.default_rng(n)
    f = np.float32
    means = torch.from_numpy(rng.uniform(-1, 1, (n, 2)).astype(f)).cuda()
    depths = np.sort(rng.uniform(0, 1, n)).astype(f)
    big = {"few": np.zeros(n, bool), "all": np.ones(n, bool),
           "turns": (np.arange(n) // 700) % 5 == 1}[kind]
    scales = np.where(big, 400.0, 0.6).astype(f)
    perm = rng.permutation(n)
    scales = torch.from_numpy(np.repeat(scales[perm, None], 2, 1).copy()).cuda()
    rot = torch.zeros(n, device="cuda")
    xys, _, radii, conics, _ = G.project_forward(means, scales, rot, H, W, BX, BY)
    d = torch.from_numpy(depths[perm].copy()).cuda()
    b = G.bin_gaussians(xys, conics, radii, d, H, W, BX, BY)
    ids, bins, _ = O.gs_bin(*(t.cpu().numpy() for t in (xys, conics, radii, d)), H, W, BX, BY)
    np.testing.assert_array_equal(b.tile_bins.cpu().numpy(), bins)
    np.testing.assert_array_equal(b.gaussian_ids_sorted.cpu().numpy(), ids)
