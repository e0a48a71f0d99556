"""What the compositing forward's segments hold: nothing where no backward can follow."""
import numpy as np
import pytest
import torch

from jax_gs_amd.renderer import rasterizer, rasterizer_tpu

pytestmark = pytest.mark.gpu
F32 = np.float32


def _scene(cuda, n, w, h, seed=0):
    rng = np.random.default_rng(seed)
    means = (rng.uniform(0, 1, (n, 2)) * [w, h]).astype(F32)
    cov = np.zeros((n, 2, 2), F32)
    cov[:, 0, 0], cov[:, 1, 1] = rng.uniform(2, 60, n), rng.uniform(2, 60, n)
    radii = np.ceil(3 * np.sqrt(cov.max((1, 2)))).astype(F32)
    arrays = (means, cov, rng.normal(0, 1, (n, 1)).astype(F32), rng.uniform(0, 1, (n, 3)).astype(F32))
    t = [torch.from_numpy(a).to(cuda) for a in arrays]
    z = torch.from_numpy(rng.uniform(1, 9, n).astype(F32)).to(cuda)
    tiles, gids, _ = rasterizer.get_tile_interactions(t[0], torch.from_numpy(radii).to(cuda),
                                                      torch.ones(n, dtype=torch.bool, device=cuda), z, h, w)
    return t, tiles, gids


@pytest.mark.parametrize("entry", [rasterizer.render_tiles, rasterizer_tpu.render_tiles_tpu])
def test_render_tiles_without_grad_mode_leaves_no_segments(cuda, entry):
    w, h = 640, 512
    t, tiles, gids = _scene(cuda, 400, w, h)
    for a in t:
        a.requires_grad_(True)
    image = entry(*t, tiles, gids, h, w)
    torch.cuda.synchronize()
    segments = rasterizer.new_segments(h, w, cuda).numel()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    with torch.no_grad():
        shown = entry(*t, tiles, gids, h, w)
    torch.cuda.synchronize()
    assert torch.cuda.max_memory_allocated() - before < segments / 4
    assert torch.equal(shown, image.detach())
