"""What the compositing forward's segments hold: nothing where no backward can follow, and no more
than the list's capacity asks for."""
import numpy as np
import pytest
import torch

from gpu_helpers import np_, rel
from jax_gs_amd import _lib, render, scenes
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


# tiles wide, tiles high, entries per tile (cycled): units of 64 (below 2048 tiles) and 128 entries
@pytest.mark.parametrize("tx,ty,counts", [
    (1, 1, [700]), (3, 2, [0, 63, 64, 65, 1, 128]), (5, 4, [1025, 0, 0, 0, 0, 2049, 4100]), (25, 21, [130, 0, 64, 700]),
    (64, 32, [128, 0, 129, 1, 300]), (90, 60, [0, 40, 0, 1300])])
def test_packed_slots_give_the_gradients_of_fixed_ones(cuda, tx, ty, counts):
    """The list as long as its entries (the tiles' slots one after another) against the same list
    with room for 4096 entries per tile (slots at fixed places); nothing is written past the
    smaller buffer."""
    T, w, h = tx * ty, 16 * tx - 3, 16 * ty - 5
    rng = np.random.default_rng(T)
    n, per = max(counts), np.resize(counts, T)
    means = rng.uniform(-4.0, 20.0, (n, 2)) + 8.0 * np.array([tx, ty])
    cov = np.zeros((n, 2, 2), F32)
    s = max(w, h) * rng.uniform(0.3, 2.0, (n, 2))
    cov[:, 0, 0], cov[:, 1, 1] = s[:, 0] ** 2, s[:, 1] ** 2
    opac = (-5.5 + rng.normal(0, 0.3, (n, 1))).astype(F32)
    col = rng.uniform(0, 1, (n, 3)).astype(F32)
    rec = rasterizer.composite_records(*[torch.from_numpy(a).to(cuda) for a in (means.astype(F32), cov, opac, col)])
    tiles = torch.from_numpy(np.repeat(np.arange(T), per).astype(np.int32)).to(cuda)
    gids = torch.from_numpy(np.concatenate([np.arange(c) for c in per]).astype(np.int32)).to(cuda)
    ranges = rasterizer.tile_ranges(tiles, T)
    room = torch.zeros(4096 * T, dtype=torch.int32, device=cuda)
    room[:gids.shape[0]] = gids
    bg = torch.tensor([0.3, 0.1, 0.6], device=cuda)
    cot = torch.from_numpy(rng.normal(0, 1, (h, w, 3)).astype(F32)).to(cuda)
    out = []
    for lst in (gids, room):
        size = rasterizer.new_segments(h, w, cuda, lst.shape[0]).numel()
        buf = torch.full((size + 65536,), 0xAB, dtype=torch.uint8, device=cuda)
        segs = buf[:size]
        image, fT, nc, _ = rasterizer.composite(rec, lst, ranges, h, w, bg, segments=segs)
        grec, gbg = torch.empty((n, 12), device=cuda), torch.empty(3, device=cuda)
        _lib.call("gs_composite_bwd_seg", _lib.stream_handle(cuda), n, _lib.ptr(rec), _lib.ptr(lst), lst.shape[0],
                  _lib.ptr(ranges), w, h, _lib.ptr(bg), _lib.ptr(cot), None, None, None, _lib.ptr(fT), _lib.ptr(nc),
                  _lib.ptr(segs), _lib.ptr(grec), _lib.ptr(gbg), 0, None, None)
        assert bool((buf[size:] == 0xAB).all())
        out.append((size, image, fT, nc, np_(grec), np_(gbg)))
    (a, b) = out
    assert a[0] < b[0] == rasterizer.new_segments(h, w, cuda).numel()
    assert all(torch.equal(x, y) for x, y in zip(a[1:4], b[1:4]))
    # the same terms, added by atomics in another order
    assert rel(a[4], b[4]) <= 2e-5 and rel(a[5], b[5]) <= 1e-4


def test_live_renders_of_a_small_scene_hold_little(cuda):
    """Three renders of 2000 Gaussians at 1440x1079 before any backward: each holds its images, its
    list (256 entries per Gaussian) and the segments of that many entries, not the 401 MB of lists of
    4096 entries in every tile."""
    sc = scenes.make_scene(1, n=2000, width=1440, height=1079)
    g, cam, _, m = scenes.to_torch(sc, cuda)
    g.means.requires_grad_(True)
    held, live = [], []
    for _ in range(3):
        before = torch.cuda.memory_allocated()
        live.append(render(g, cam, mask=m, sh_degree=sc["sh_degree"])[0])
        held.append(torch.cuda.memory_allocated() - before)
    assert max(held) < 100e6, held
    sum(i.sum() for i in live).backward()
    assert bool(torch.isfinite(g.means.grad).all())


def test_composite_refuses_segments_of_another_size(cuda):
    """A buffer made for a smaller image or a shorter list, or on the host, is refused before the
    launch that would write past it."""
    w, h, n = 200, 120, 300
    t, tiles, gids = _scene(cuda, n, w, h)
    rec = rasterizer.composite_records(*t)
    ranges = rasterizer.tile_ranges(tiles, ((w + 15) // 16) * ((h + 15) // 16))
    bg = torch.zeros(3, device=cuda)
    length = gids.shape[0]
    good = rasterizer.new_segments(h, w, cuda, length)
    for bad in (rasterizer.new_segments(h - 16, w, cuda, length), rasterizer.new_segments(h, w, cuda, 1000), good[:-256],
                good.cpu()):
        with pytest.raises(ValueError, match="segments must hold"):
            rasterizer.composite(rec, gids, ranges, h, w, bg, segments=bad)
    rasterizer.composite(rec, gids, ranges, h, w, bg, segments=good)
