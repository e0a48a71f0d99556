"""The forward of images from 2048 to 6143 tiles: survivors staged in LDS and walked in pairs, against
the oracle's render_tiles on hand-made lists (lengths around a pair, a batch of 64 and a segment,
pixels that close at either entry of a pair, few survivors of a batch); and the queue that a tile's
waves fill from a deferred binning's superblock words, against the list written whole (tiles with few
entries among thousands of words, with counts around a batch and the queue's lead)."""
import numpy as np
import pytest
import torch

import oracle
from gpu_helpers import np_
from jax_gs_amd import _lib
from jax_gs_amd.renderer import rasterizer

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.mark.parametrize("count", [0, 1, 2, 3, 63, 64, 65, 127, 129])
@pytest.mark.parametrize("opacity,sigma", [(-2.0, 300.0), (6.0, 300.0), (1.0, 6.0)])
def test_walk_in_pairs_equals_oracle(cuda, count, opacity, sigma):
    w, h = 1024 - 3, 528 - 9
    tx, ty = 64, 33
    rng = np.random.default_rng(1000 * count + int(10 * opacity + 100))
    n = max(count, 1)
    means = rng.uniform(-2.0, [w + 2.0, h + 2.0], (n, 2)).astype(F32)
    s = rng.uniform(0.7, 1.4, (n, 2)) * sigma
    cov = np.zeros((n, 2, 2), F32)
    cov[:, 0, 0], cov[:, 1, 1] = s[:, 0] ** 2, s[:, 1] ** 2
    cov[:, 0, 1] = cov[:, 1, 0] = rng.uniform(-0.6, 0.6, n) * s[:, 0] * s[:, 1]
    opac = (opacity + rng.normal(0, 0.5, (n, 1))).astype(F32)
    col = rng.uniform(0, 1, (n, 3)).astype(F32)
    bg = np.array([0.2, 0.5, 0.9], F32)
    tiles = np.concatenate([np.repeat(np.arange(tx * ty), count), np.full(600, tx * ty)]).astype(np.int32)
    gids = np.concatenate([np.tile(np.arange(count), tx * ty), np.zeros(600)]).astype(np.int32)
    img_o, fT_o, nc_o = oracle.render_tiles(means, cov, opac, col, tiles, gids, h, w, background=bg)
    t = [torch.from_numpy(a).to(cuda) for a in (means, cov, opac, col, tiles, gids, bg)]
    rec = rasterizer.composite_records(*t[:4])
    ranges = rasterizer.tile_ranges(t[4], tx * ty)
    img, fT, nc, _ = rasterizer.composite(rec, t[5], ranges, h, w, t[6])
    # 32-bit blending: each of up to `count` products and sums rounds at 2^-24 of a value below 1;
    # an exponent's terms reach about 50 and round at 2^-24 a few times, 1.2e-5 of an alpha, and
    # the weights of a pixel add up to at most 1
    tol = (4 + count) * 2.0 ** -24 * 4 + 2e-5
    same = np_(nc) == nc_o  # a transmittance within rounding of the threshold may end an entry apart
    assert same.mean() >= 0.995
    assert np.abs(np_(img) - img_o)[same].max() <= tol
    assert np.abs(np_(img) - img_o).max() <= tol + 1e-4
    assert np.abs(np_(fT) - fT_o)[same].max() <= tol


@pytest.mark.parametrize("counts", [[0, 1, 63, 64], [65, 127, 128, 129], [191, 192, 193, 300], [2, 640, 1500, 4200]])
@pytest.mark.parametrize("crowd", [0, 3000, 9000])
def test_queue_of_sparse_tiles_equals_whole_list(cuda, counts, crowd):
    """Tiles of one superblock: one holds `crowd` Gaussians, four others counts[k] each, spread over
    the crowd's words by depth.  All are faint, so every wave walks its list to the end."""
    w, h = 1024, 528
    rng = np.random.default_rng(sum(counts) + crowd)
    per = [(0, 0, crowd)] + [(x, y, c) for (x, y), c in zip([(1, 0), (7, 3), (4, 7), (0, 5)], counts)]
    centre = np.concatenate([np.tile([[16.0 * x + 8, 16.0 * y + 8]], (c, 1)) for x, y, c in per]
                            + [rng.uniform(200, [w, h], (50, 2))])
    n = centre.shape[0]
    order = rng.permutation(n)
    means = (centre + rng.uniform(-2, 2, (n, 2)))[order].astype(F32)
    t = [torch.from_numpy(a).to(cuda) for a in (means, np.full(n, 5.0, F32), np.ones(n, bool),
                                                rng.uniform(1, 50, n).astype(F32))]
    cov = torch.zeros((n, 2, 2), device=cuda)
    cov[:, 0, 0] = cov[:, 1, 1] = 4.0
    rec = rasterizer.composite_records(t[0], cov, torch.full((n, 1), -9.0, device=cuda), torch.rand((n, 3), device=cuda))
    bg = torch.tensor([0.1, 0.2, 0.3], device=cuda)
    full = rasterizer.bin_gaussians(*t, h, w, want_tiles=False)
    b = rasterizer.bin_gaussians(*t, h, w, want_tiles=False, deferred=True)
    assert int(b["stats"][_lib.STAT["entries_deferred"]]) == 1
    ranges = np_(full["ranges"]).astype(np.int64)
    for x, y, c in per:
        k = y * 64 + x
        assert ranges[k + 1] - ranges[k] >= c
    b["sorted_gids"].fill_(-7)
    got = rasterizer.composite(rec, b["sorted_gids"], b["ranges"], h, w, bg, bins=b,
                               segments=rasterizer.new_segments(h, w, cuda, b["capacity"]))
    want = rasterizer.composite(rec, full["sorted_gids"], full["ranges"], h, w, bg)
    for a, c in zip(got[:3], want):
        assert torch.equal(a, c)
    keep = np.concatenate([np.arange(ranges[k], min(ranges[k + 1], ranges[k] + 4096)) for k in range(64 * 33)])
    np.testing.assert_array_equal(np_(b["sorted_gids"])[keep], np_(full["sorted_gids"])[keep])
