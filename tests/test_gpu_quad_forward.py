"""The forward of images below 2048 tiles (four entries a step, 4 x 4 pixels a wave) against
the oracle's render_tiles on hand-made entry lists: list lengths around a step (4), a pair of
steps (8), a batch (64) and a chunk (512), pixels that close at each of a step's four entries,
Gaussians small enough that most 4 x 4 blocks drop them, and frames cut through a block."""
import numpy as np
import pytest
import torch

import oracle
from gpu_helpers import np_
from jax_gs_amd.renderer import rasterizer

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.mark.parametrize("count", [0, 1, 3, 4, 5, 8, 9, 63, 64, 65, 71, 129, 513, 4099])
@pytest.mark.parametrize("opacity", [-2.0, 6.0])
@pytest.mark.parametrize("w,h,sigma", [(16, 16, 40.0), (29, 35, 1.5)])
def test_quad_forward_equals_oracle(cuda, count, opacity, w, h, sigma):
    rng = np.random.default_rng(1000 * count + int(10 * opacity + 100) + w)
    n = max(count, 1)
    tx, ty = (w + 15) // 16, (h + 15) // 16
    means2d = rng.uniform(-2.0, [w + 2.0, h + 2.0], (n, 2)).astype(F32)
    s = rng.uniform(0.7, 1.4, (n, 2)) * sigma
    cov = np.zeros((n, 2, 2), F32)
    cov[:, 0, 0], cov[:, 1, 1] = s[:, 0] ** 2, s[:, 1] ** 2
    cov[:, 0, 1] = cov[:, 1, 0] = rng.uniform(-0.6, 0.6, n) * s[:, 0] * s[:, 1]
    opac = (opacity + rng.normal(0, 0.5, (n, 1))).astype(F32)
    col = rng.uniform(0, 1, (n, 3)).astype(F32)
    bg = np.array([0.2, 0.5, 0.9], F32)
    # every tile holds the same `count` entries, then 600 empty slots (no clamped chunk)
    tiles = np.concatenate([np.repeat(np.arange(tx * ty), count), np.full(600, tx * ty)]).astype(np.int32)
    gids = np.concatenate([np.tile(np.arange(count), tx * ty), np.zeros(600)]).astype(np.int32)
    img_o, fT_o, nc_o = oracle.render_tiles(means2d, cov, opac, col, tiles, gids, h, w, background=bg)
    t = [torch.from_numpy(a).to(cuda) for a in (means2d, cov, opac, col, tiles, gids, bg)]
    rec = rasterizer.composite_records(*t[:4])
    ranges = rasterizer.tile_ranges(t[4], tx * ty)
    img, fT, nc, _ = rasterizer.composite(rec, t[5], ranges, h, w, t[6])
    # 32-bit blending: each of up to 4096 products and sums rounds at 2^-24 of a value below 1
    tol = (4 + min(count, 4096)) * 2.0 ** -24 * 4
    assert np.abs(np_(img) - img_o).max() <= tol + 1e-4 * (np_(nc) != nc_o).any()
    same = np_(nc) == nc_o  # a transmittance within rounding of the threshold may end an entry apart
    assert same.mean() >= 0.995
    assert np.abs(np_(fT) - fT_o)[same].max() <= tol
