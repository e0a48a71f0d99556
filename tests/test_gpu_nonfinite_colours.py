"""A colour that is not finite reaches only the pixels that its Gaussian reaches, in frames below 2048
tiles: 4 x 4 pixels a wave in the forward, and in the backward one pixel a lane (below 512 tiles) or
four, whose first is evaluated whether or not the entry reaches it."""
import numpy as np
import pytest
import torch

from gpu_helpers import np_
from jax_gs_amd.renderer import rasterizer

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.mark.parametrize("tx,ty", [(6, 5), (25, 21), (46, 44)])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
def test_infinite_colours_stay_where_they_are(cuda, tx, ty, value):
    w, h = 16 * tx - 3, 16 * ty - 5
    rng = np.random.default_rng(tx)
    n = 100 + 2 * tx * ty
    odd = np.arange(n) % 40 == 7  # about one in a 64-entry batch
    means = (rng.uniform(0, 1, (n, 2)) * [w, h]).astype(F32)
    cov = np.zeros((n, 2, 2), F32)
    s = rng.uniform(1.0, 3.0, (n, 2))
    s[odd] = 1.2
    cov[:, 0, 0], cov[:, 1, 1] = s[:, 0] ** 2, s[:, 1] ** 2
    radii = np.ceil(5 * s.max(1)).astype(F32)  # past the gate at 4.5 sigma
    z = rng.uniform(1, 9, n).astype(F32)
    opac = rng.normal(0, 1, (n, 1)).astype(F32)
    col = rng.uniform(0, 1, (n, 3)).astype(F32)
    t = [torch.from_numpy(a).to(cuda) for a in (means, cov, opac, col)]
    tiles, gids, _ = rasterizer.get_tile_interactions(t[0], torch.from_numpy(radii).to(cuda),
                                                      torch.ones(n, dtype=torch.bool, device=cuda),
                                                      torch.from_numpy(z).to(cuda), h, w)
    # pixels that an odd Gaussian's gate (power > -10) reaches; and a margin in which none is compared
    ys, xs = np.mgrid[0:h, 0:w] + 0.5
    hit = np.zeros((h, w), bool)
    for k in np.nonzero(odd)[0]:
        power = -0.5 * (((xs - means[k, 0]) / s[k, 0]) ** 2 + ((ys - means[k, 1]) / s[k, 1]) ** 2)
        hit |= power > -10.001
    assert 0.01 < hit.mean() < 0.5
    cot = torch.from_numpy(rng.normal(0, 1, (h, w, 3)).astype(F32) * ~hit[:, :, None]).to(cuda)
    res = []
    for c in (0.25, value):
        leaves = [a.clone().requires_grad_(True) for a in t]
        with torch.no_grad():
            leaves[3][torch.from_numpy(odd).to(cuda)] = float(c)
        image = rasterizer.render_tiles(*leaves, tiles, gids, h, w)
        image.backward(cot)
        res.append((np_(image), [np_(a.grad) for a in leaves]))
    (image, grads), (image_o, grads_o) = res
    np.testing.assert_array_equal(image[~hit], image_o[~hit])
    assert np.isfinite(image_o).all() == False and np.isfinite(image).all()  # noqa: E712
    # Gaussians that share no pixel with an odd one: a distance of both gates
    d = np.linalg.norm(means[:, None] - means[None, odd], axis=2) - 4.6 * (s.max(1)[:, None] + 1.2)
    apart = (d > 0).all(1) & ~odd
    assert apart.sum() > 50
    for a, b in zip(grads, grads_o):
        assert np.isfinite(b[apart]).all()
        # the same terms, added by atomics in another order
        np.testing.assert_allclose(a[apart], b[apart], rtol=1e-3, atol=1e-5 * np.abs(a[apart]).max())
