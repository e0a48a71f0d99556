"""The binning's one-workgroup scan over the tiles and its statistics at the edges of its rounds
(8192 tiles) and waves, and the background's cotangent at the edges of its blocks (2048 pixels, four
of them in flight per lane)."""
import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tx, ty", [(1, 1), (7, 9), (64, 1), (1, 65), (128, 64), (2, 4095), (2731, 3), (181, 91)])
def test_ranges_and_statistics(cuda, tx, ty):
    from jax_gs_amd import _lib
    from jax_gs_amd.renderer import rasterizer

    rng = np.random.default_rng(tx * 10007 + ty)
    n, W, H = 1500, 16 * tx - 3, 16 * ty - 5
    means2d = (rng.uniform(-0.1, 1.1, (n, 2)) * [W, H]).astype(np.float32)
    means2d[: n // 2] = means2d[0]  # one tile with more than a chunk of entries
    radii = np.ceil(rng.uniform(0, 40, n)).astype(np.float32)
    valid = rng.uniform(size=n) < 0.9
    depths = rng.uniform(-0.5, 20, n).astype(np.float32)
    b = rasterizer.bin_gaussians(*[torch.from_numpy(a).to(cuda) for a in (means2d, radii, valid, depths)], H, W)
    st_o, _, n_o = oracle.tile_interactions(means2d, radii, valid, depths, H, W)
    T = tx * ty
    counts = np.bincount(st_o[(st_o >= 0) & (st_o < T)], minlength=T)
    np.testing.assert_array_equal(b["ranges"].cpu().numpy(), np.concatenate([[0], np.cumsum(counts)]))
    S, st = _lib.STAT, b["stats"].cpu().numpy()
    assert st[S["n_interactions"]] == n_o
    assert st[S["max_interactions_per_tile"]] == counts.max()
    assert st[S["overflow_tiles"]] == (counts > 512).sum()
    assert st[S["overflow_interactions"]] == np.maximum(counts - 512, 0).sum()
    assert st[S["truncated_tiles"]] == (counts > 4096).sum()


@pytest.mark.parametrize("H, W", [(1, 1), (1, 255), (2, 1024), (2, 1025), (64, 33), (1030, 1024)])
def test_background_cotangent(cuda, H, W):
    """Without Gaussians the image is the background: its cotangent is the image cotangent's sum."""
    from jax_gs_amd import Camera, Gaussians, render

    e = [torch.zeros(s, device=cuda) for s in ((1, 3), (1, 3), (1, 4), (1, 1), (1, 1, 3))]
    e[0][0, 2] = -5.0  # behind the camera
    e[2][0, 0] = 1.0
    eye = torch.eye(4, device=cuda)
    bg = torch.tensor([0.2, 0.5, 0.7], device=cuda, requires_grad=True)
    image, _ = render(Gaussians(*e), Camera(W, H, 50.0, 50.0, W / 2, H / 2, eye, eye), background=bg)
    cot = torch.rand((H, W, 3), generator=torch.Generator(device=cuda).manual_seed(H * W), device=cuda)
    image.backward(cot)
    want = cot.double().sum((0, 1))
    # a lane adds up to H W / (256 * blocks) terms, then trees and one atomic per block
    assert ((bg.grad.double() - want).abs() <= 1e-5 * want).all()
