"""Kernels over the reference's full tile arrays: the pass that finds the tiles' ranges (groups of
four entries, a scalar path where the array is not 16-byte aligned or ends inside a group) and the
fill of the arrays (several workgroups per span of 1024 Gaussians)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ranges(tiles, T):
    """ranges[t] = the first entry whose tile is >= t (the arrays are sorted)."""
    return np.searchsorted(tiles, np.arange(T + 1), side="left")


@pytest.mark.parametrize("offset", [0, 1, 2, 3])
@pytest.mark.parametrize("length", [1, 3, 4, 5, 511, 4096, 2 * 2048 * 256 * 4 * 4 + 3])
def test_tile_ranges_alignment_and_remainders(cuda, length, offset):
    from jax_gs_amd.renderer import rasterizer

    rng = np.random.default_rng(length + offset)
    T = 37
    # -1 slots first, T sentinels last, some tiles empty, boundaries anywhere in a group
    tiles = np.sort(rng.choice(np.array([-1, 0, 1, 2, 5, 6, 7, 20, 21, 36, T]), length)).astype(np.int32)
    base = torch.zeros(length + offset, dtype=torch.int32, device=cuda)
    base[offset:] = torch.from_numpy(tiles).to(cuda)
    got = rasterizer.tile_ranges(base[offset:], T).cpu().numpy()
    np.testing.assert_array_equal(got, _ranges(tiles, T))


@pytest.mark.parametrize("n", [63, 64, 65, 1023, 1024, 1025, 2113])
def test_reference_arrays_at_the_spans_edges(cuda, n):
    import oracle
    from jax_gs_amd.renderer import rasterizer

    rng = np.random.default_rng(n)
    W, H = 120, 90
    means2d = rng.uniform(-40, 160, (n, 2)).astype(np.float32)
    radii = np.ceil(rng.uniform(0, 40, n)).astype(np.float32)
    valid = rng.uniform(size=n) < 0.8
    depths = rng.uniform(-2.0, 20, n).astype(np.float32)
    st, sg, count = rasterizer.get_tile_interactions(*[torch.from_numpy(a).to(cuda) for a in
                                                       (means2d, radii, valid, depths)], H, W)
    st_o, sg_o, n_o = oracle.tile_interactions(means2d, radii, valid, depths, H, W)
    assert int(count) == n_o
    np.testing.assert_array_equal(st.cpu().numpy(), st_o)
    np.testing.assert_array_equal(sg.cpu().numpy(), sg_o)
