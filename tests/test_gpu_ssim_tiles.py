"""The L1 + SSIM kernels at the edges of their tiles (8 rows x 116 columns, groups of four columns
that are read and stored whole at any address but for a row's last, shorter one): means and image
gradient against the float64 oracle."""
import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H, W, C", [(1, 1, 3), (1, 116, 1), (8, 4, 3), (7, 115, 2), (8, 116, 3), (9, 117, 3),
                                     (3, 121, 4), (16, 128, 4), (13, 111, 3), (17, 232, 2), (5, 236, 3)])
@pytest.mark.parametrize("shift", [0, 1])
def test_l1_ssim_tile_edges(cuda, H, W, C, shift):
    """`shift` moves the images and the gradient off 16-byte alignment by one value."""
    from jax_gs_amd import _lib

    rng = np.random.default_rng(1000 * H + 10 * W + C)
    shape, count = (H, W, C), H * W * C
    tgt = rng.uniform(0, 1, shape).astype(np.float32)
    pred = np.clip(tgt + rng.normal(0, 0.2, shape), 0, 1).astype(np.float32)

    def put(a):
        b = torch.full((count + 2,), float("nan"), device=cuda)
        b[shift:shift + count] = torch.from_numpy(a.ravel()).to(cuda)
        return b

    p, t, grad = put(pred), put(tgt), put(np.zeros(shape, np.float32))
    gout = torch.tensor([0.8, -0.1], device=cuda)
    nb = _lib.lib().gs_l1_ssim_workspace_size(H, W, C)
    ws = torch.empty((nb,), dtype=torch.uint8, device=cuda)
    out = torch.empty((2,), device=cuda)
    s = _lib.stream_handle(cuda)
    at = [b[shift:] for b in (p, t, grad)]
    _lib.call("gs_l1_ssim", s, H, W, C, _lib.ptr(at[0]), _lib.ptr(at[1]), _lib.ptr(out), 1, _lib.ptr(ws), nb)
    _lib.call("gs_l1_ssim_bwd", s, H, W, C, _lib.ptr(at[0]), _lib.ptr(at[1]), _lib.ptr(gout), _lib.ptr(ws), nb,
              _lib.ptr(at[2]))
    # nothing is written beside the gradient
    g = grad.cpu().numpy()
    assert np.isnan(g[:shift]).all() and np.isnan(g[shift + count:]).all()
    want_l1, seed = oracle.l1_loss_and_grad(pred, tgt)
    l1, ssim = out.cpu().numpy()
    assert abs(l1 - want_l1) <= 1e-6 * want_l1 + 1e-9
    assert abs(ssim - oracle.ssim(pred, tgt)) <= 1e-5
    want = 0.8 * seed.astype(np.float64) + oracle.ssim_vjp(pred, tgt, -0.1)
    got = g[shift:shift + count].reshape(shape)
    assert np.linalg.norm(got - want) <= 1e-4 * np.linalg.norm(want)


@pytest.mark.parametrize("which", [(1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 1)])
@pytest.mark.parametrize("lam", [0.2, 0.0, 1])
def test_l1_ssim_loss_and_cotangents(cuda, lam, which):
    """l1_ssim_loss's three outputs and the gradient from any of their cotangents against the
    composition of l1_and_ssim: the outputs' bits, the gradient to float32 rounding of its two
    scalar cotangents."""
    from jax_gs_amd.training import losses

    rng = np.random.default_rng(3)
    t = torch.from_numpy(rng.uniform(0, 1, (21, 130, 3)).astype(np.float32)).to(cuda)
    p0 = (t + 0.1 * torch.from_numpy(rng.normal(0, 1, t.shape).astype(np.float32)).to(cuda)).clamp(0, 1)
    outs, grads = [], []
    for fused in (True, False):
        p = p0.clone().requires_grad_(True)
        if fused:
            o = losses.l1_ssim_loss(p, t, lam)
        else:
            l1, s = losses.l1_and_ssim(p, t)
            d = losses._d_ssim(s)
            o = ((1.0 - lam) * l1 + lam * d, l1, d)
        sum(w * (k + 1.5) * v for k, (w, v) in enumerate(zip(which, o)) if w).backward()
        outs.append([float(v.detach()) for v in o])
        grads.append(p.grad)
    assert outs[0] == outs[1]
    scale = grads[1].norm()
    assert (grads[0] - grads[1]).norm() <= 1e-6 * scale if scale > 0 else not grads[0].any()


def test_l1_ssim_loss_of_equal_images(cuda):
    """At SSIM = 1 the max ties or rounds: the gradient follows torch.maximum's half."""
    from jax_gs_amd.training import losses

    t = torch.rand((40, 50, 3), device=cuda)
    grads = []
    for fused in (True, False):
        p = t.clone().requires_grad_(True)
        l1, s = (None, None) if fused else losses.l1_and_ssim(p, t)
        total = losses.l1_ssim_loss(p, t)[0] if fused else 0.8 * l1 + 0.2 * losses._d_ssim(s)
        total.backward()
        grads.append(p.grad)
    assert (grads[0] - grads[1]).norm() <= 1e-6 * grads[1].norm() + 1e-12
