"""The compositing VJP over segments (gs_composite_fwd_seg, gs_composite_bwd_seg) against the
walk of whole lists (gs_composite_fwd, gs_composite_bwd) on hand-made entry lists: lengths at
the ends of segments of every unit, transparent lists that every pixel walks to the end and
opaque ones that close inside a segment, and so many pieces that the units are coarsened to fit
the launch; the builds change at 512, 2048 and 6144 tiles (at 6144 lists have no segments)."""
import numpy as np
import pytest
import torch

from gpu_helpers import np_, rel
from jax_gs_amd import _lib
from jax_gs_amd.renderer import rasterizer

pytestmark = pytest.mark.gpu
F32 = np.float32


# tiles wide, tiles high, entries per tile (cycled over the tiles), opacity logit
@pytest.mark.parametrize("tx,ty,counts,opacity", [
    (1, 1, [4096], -5.0), (1, 1, [1], 0.0), (2, 3, [63, 64, 65, 0, 128, 129], -4.0),
    (3, 2, [1023, 1024, 1025, 2048, 2049, 5000], -6.5), (4, 4, [700, 1200, 300, 40], 1.0),
    (25, 25, [4096], -6.5), (40, 13, [4096, 2000, 65, 512], -6.0), (64, 32, [500, 128, 129, 1100], -5.0),
    (90, 60, [1300, 260, 10], -5.5), (128, 48, [200, 600], -5.0)])
@pytest.mark.parametrize("window", [False, True])
def test_segments_equal_whole_walks(cuda, tx, ty, counts, opacity, window):
    T, w, h = tx * ty, 16 * tx - 3, 16 * ty - 5
    rng = np.random.default_rng(T + len(counts))
    n, per = max(counts), np.resize(counts, T)
    # Gaussians around one tile's centre, shifted to each tile: ids repeat over the tiles
    m = 2
    base = rng.uniform(-4.0, 20.0, (n, 2))
    means2d = np.concatenate([base + 16.0 * np.array([(k * 7) % tx, (k * 5) % ty]) for k in range(m)]).astype(F32)
    s = rng.uniform(3.0, 40.0, (n * m, 2))
    cov = np.zeros((n * m, 2, 2), F32)
    cov[:, 0, 0], cov[:, 1, 1] = s[:, 0] ** 2, s[:, 1] ** 2
    opac = (opacity + rng.normal(0, 0.3, (n * m, 1))).astype(F32)
    col = rng.uniform(0, 1, (n * m, 3)).astype(F32)
    tiles = np.repeat(np.arange(T), per)
    gids = np.concatenate([np.arange(c) + n * (t % m) for t, c in enumerate(per)] + [np.zeros(0)])
    tail = 0 if window else 600
    tiles = np.concatenate([tiles, np.full(tail, T)]).astype(np.int32)
    gids = np.concatenate([gids, np.zeros(tail)]).astype(np.int32)
    t = [torch.from_numpy(a).to(cuda) for a in (means2d, cov, opac, col, tiles, gids)]
    bg = torch.tensor([0.3, 0.1, 0.6], device=cuda)
    cot = torch.from_numpy(rng.normal(0, 1, (h, w, 3)).astype(F32)).to(cuda)
    rec = rasterizer.composite_records(*t[:4])
    ranges = rasterizer.tile_ranges(t[4], T)
    win = rasterizer.window_from_list(t[5]) if window else None
    segs = rasterizer.new_segments(h, w, cuda).fill_(0xFF)
    image, fT, nc, order = rasterizer.composite(rec, t[5], ranges, h, w, bg, window=win)
    image_s, fT_s, nc_s, _ = rasterizer.composite(rec, t[5], ranges, h, w, bg, window=win, segments=segs)
    assert torch.equal(image, image_s) and torch.equal(fT, fT_s) and torch.equal(nc, nc_s)
    N = rec.shape[0]
    head = (_lib.stream_handle(cuda), N, _lib.ptr(rec), _lib.ptr(t[5]), t[5].shape[0], _lib.ptr(ranges), w, h,
            _lib.ptr(bg), _lib.ptr(cot))
    out = []
    for seg in (False, True):
        grec, gbg = torch.empty((N, 12), device=cuda), torch.empty(3, device=cuda)
        tail_args = (_lib.ptr(grec), _lib.ptr(gbg), 0, _lib.ptr(win), None)
        if seg:
            _lib.call("gs_composite_bwd_seg", *head, None, None, None, _lib.ptr(fT), _lib.ptr(nc), _lib.ptr(segs),
                      *tail_args)
        else:
            _lib.call("gs_composite_bwd", *head, _lib.ptr(fT), _lib.ptr(nc), _lib.ptr(order), *tail_args)
        out.append((np_(grec), np_(gbg)))
    # the whole walk recovers T over up to 4096 divisions, each rounded at 2^-24; sums of both
    # signs over the pixels cancel to a part of their terms (8 covers it with margin)
    tol = 8 * (64 + n) * 2.0 ** -24
    assert rel(out[1][0], out[0][0]) <= tol
    assert np.array_equal(out[1][0] == 0, out[0][0] == 0) or rel(out[1][0], out[0][0]) <= 1e-5
    assert rel(out[1][1], out[0][1]) <= 1e-4


@pytest.mark.parametrize("w,h", [(128, 96), (504, 378), (1280, 720)])
def test_segments_of_records_beyond_4gib(cuda, w, h):
    """A walked record is addressed by its byte offset in a 32-bit register while the records span
    less than 4 GiB, and by its id beyond: the same scene at the end of 4.3 GB of records, one
    pixel per lane, four, and four from 2048 tiles on."""
    from jax_gs_amd import scenes
    from jax_gs_amd.renderer.projection import preprocess

    sc = scenes.make_scene(2, n=20000, width=w, height=h)
    g, cam, _, mask = scenes.to_torch(sc, cuda)
    n_big = (2 ** 32 - 64) // (4 * _lib.GS_REC_STRIDE) + 1
    with torch.no_grad():
        pre = preprocess(g, cam, mask=mask, sh_degree=sc["sh_degree"])
        b = rasterizer.bin_gaussians(pre["means2d"], pre["radii"], pre["valid"], pre["depths"], h, w,
                                     want_tiles=False)
    rec, gids, ranges = pre["records"], b["sorted_gids"], b["ranges"]
    n = rec.shape[0]
    big = torch.empty((n_big, _lib.GS_REC_STRIDE), device=cuda)
    big[n_big - n:] = rec
    bg = torch.tensor([0.1, 0.2, 0.3], device=cuda)
    cot = torch.rand((h, w, 3), generator=torch.Generator(device=cuda).manual_seed(3), device=cuda)
    images, grads = [], []
    for rr, gg in ((rec, gids), (big, gids + (n_big - n))):
        segs = rasterizer.new_segments(h, w, cuda, gg.shape[0])
        image, fT, nc, _ = rasterizer.composite(rr, gg, ranges, h, w, bg, segments=segs)
        grec = torch.empty_like(rr)
        _lib.call("gs_composite_bwd_seg", _lib.stream_handle(cuda), rr.shape[0], _lib.ptr(rr), _lib.ptr(gg),
                  gg.shape[0], _lib.ptr(ranges), w, h, _lib.ptr(bg), _lib.ptr(cot), None, None, None, _lib.ptr(fT),
                  _lib.ptr(nc), _lib.ptr(segs), _lib.ptr(grec), None, 0, None, None)
        images.append(image)
        grads.append(np_(grec[-n:]))
        assert not grec[:-n].any()
    assert torch.equal(*images) and np.abs(grads[0]).max() > 0
    # the same terms, added by atomics in another order
    assert rel(grads[1], grads[0]) <= 1e-5
