"""The forward of mid-size images gives a tile two waves of eight rows.  Where the image ends in
the upper half of its last tile row (1 to 8 rows of it), the lower waves hold no pixel and must walk
nothing: not a tile's list, nor its superblock's words."""
import numpy as np
import pytest
import torch

from gpu_helpers import np_, rel
from jax_gs_amd import _lib
from jax_gs_amd.renderer import rasterizer

pytestmark = pytest.mark.gpu
F32 = np.float32
TX, TY = 64, 34  # 2176 tiles


def _wide(cuda, w, h):
    """Two Gaussians far wider than the image: an opaque one (id 0) and a faint one (id 1)."""
    means = torch.tensor([[w / 2, h / 2]] * 2, device=cuda)
    cov = torch.zeros((2, 2, 2), device=cuda)
    cov[:, 0, 0] = cov[:, 1, 1] = 5000.0 ** 2
    opac = torch.tensor([[8.0], [-6.0]], device=cuda)
    col = torch.tensor([[0.2, 0.5, 0.8], [0.9, 0.4, 0.1]], device=cuda)
    return rasterizer.composite_records(means, cov, opac, col)


@pytest.mark.parametrize("rows", [1, 8, 9, 16])
def test_waves_below_the_image_do_not_walk(cuda, rows):
    """The tile order ranks the tiles by the longer of their waves' walks: 200 entries in the upper
    tile rows, while the last row's waves are opaque within the first batch of their 1024."""
    w, h, T = 16 * TX, 16 * (TY - 1) + rows, TX * TY
    last = np.arange(T) >= T - TX
    per = np.where(last, 1024, 200)
    tiles = np.concatenate([np.repeat(np.arange(T), per), np.full(600, T)]).astype(np.int32)
    gids = np.concatenate([np.repeat(np.where(last, 0, 1), per), np.zeros(600)]).astype(np.int32)
    rec = _wide(cuda, w, h)
    g = torch.from_numpy(gids).to(cuda)
    ranges = rasterizer.tile_ranges(torch.from_numpy(tiles).to(cuda), T)
    bg = torch.tensor([0.3, 0.1, 0.6], device=cuda)
    image, fT, nc, order = rasterizer.composite(rec, g, ranges, h, w, bg)
    order = np_(order)
    np.testing.assert_array_equal(np.sort(order), np.arange(T))
    assert not last[order[:T - TX]].any()
    # the same frame with segments, and its gradients against the walk of whole lists
    segs = rasterizer.new_segments(h, w, cuda).fill_(0xFF)
    image_s, fT_s, nc_s, _ = rasterizer.composite(rec, g, ranges, h, w, bg, segments=segs)
    assert torch.equal(image, image_s) and torch.equal(fT, fT_s) and torch.equal(nc, nc_s)
    cot = torch.rand((h, w, 3), generator=torch.Generator(device=cuda).manual_seed(rows), device=cuda)
    head = (_lib.stream_handle(cuda), 2, _lib.ptr(rec), _lib.ptr(g), g.shape[0], _lib.ptr(ranges), w, h, _lib.ptr(bg),
            _lib.ptr(cot))
    tail = (None, 0, None, None)
    whole, seg = torch.empty((2, 12), device=cuda), torch.empty((2, 12), device=cuda)
    o = torch.from_numpy(order).to(cuda)
    _lib.call("gs_composite_bwd", *head, _lib.ptr(fT), _lib.ptr(nc), _lib.ptr(o), _lib.ptr(whole), *tail)
    _lib.call("gs_composite_bwd_seg", *head, None, None, None, _lib.ptr(fT), _lib.ptr(nc), _lib.ptr(segs),
              _lib.ptr(seg), *tail)
    # half a million pixels' terms per value, added by atomics in another order
    assert rel(np_(seg)[:, 5:9], np_(whole)[:, 5:9]) <= 1e-4


@pytest.mark.parametrize("rows", [1, 8])
def test_waves_below_the_image_queue_no_words(cuda, rows):
    """With a deferred list a wave stores the ids it queues.  The last row's tiles hold 1500 opaque
    Gaussians there: the upper wave is done within the first batches, so most ids stay unwritten."""
    w, h, T = 16 * TX, 16 * (TY - 1) + rows, TX * TY
    rng = np.random.default_rng(rows)
    n, dense = 4000, 1500
    means = (rng.uniform(0, 1, (n, 2)) * [w, h]).astype(F32)
    means[:dense] = [w / 2 + 0.5, h - 0.5] + rng.uniform(-2, 2, (dense, 2))
    radii = np.full(n, 30.0, F32)
    depths = rng.uniform(5, 20, n).astype(F32)
    depths[:dense] = rng.uniform(1, 2, dense)
    cov = np.zeros((n, 2, 2), F32)
    cov[:, 0, 0] = cov[:, 1, 1] = 100.0
    t = [torch.from_numpy(a).to(cuda) for a in (means, radii, np.ones(n, bool), depths)]
    rec = rasterizer.composite_records(t[0], torch.from_numpy(cov).to(cuda), torch.full((n, 1), 8.0, device=cuda),
                                       torch.rand((n, 3), device=cuda))
    bg = torch.zeros(3, device=cuda)
    full = rasterizer.bin_gaussians(*t, h, w, want_tiles=False)
    b = rasterizer.bin_gaussians(*t, h, w, want_tiles=False, deferred=True)
    assert int(b["stats"][_lib.STAT["entries_deferred"]]) == 1
    b["sorted_gids"].fill_(-7)
    out = rasterizer.composite(rec, b["sorted_gids"], b["ranges"], h, w, bg, bins=b,
                               segments=rasterizer.new_segments(h, w, cuda))
    want = rasterizer.composite(rec, full["sorted_gids"], full["ranges"], h, w, bg)
    for a, c in zip(out[:3], want):
        assert torch.equal(a, c)
    tile = T - TX + TX // 2
    start, end = (int(v) for v in b["ranges"][tile:tile + 2])
    ids = np_(b["sorted_gids"])[start:end]
    assert end - start >= dense
    # the batch walked, the one fetched ahead and the queue's lead
    assert (ids != -7).sum() <= 256
    met = int(want[2][h - rows:, 16 * (TX // 2):16 * (TX // 2) + 16].max())
    np.testing.assert_array_equal(ids[:met], np_(full["sorted_gids"])[start:start + met])
