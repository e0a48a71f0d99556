"""The workloads whose speed this package is judged by, one dict of plain values each.

Every case is what a program that uses the package has it do: a viewer's frames (``render``),
steps that fit the Gaussians to a photograph (``render_l1`` and its backward, ``train_step``,
the photometric loss on its own), the refinement of a camera, and the module functions called
one by one.  ``prepare`` makes what such a program holds before the call, ``run`` is one pass
through the public entry points, ``exact`` is the same result in 64 bits from plain torch.

The synthetic scenes follow the distributions of ``jax_gs_amd.scenes`` (clusters of Gaussians
in front of the camera, log-normal sizes, normally distributed opacity logits), drawn on the
GPU so that they are made quickly.
"""
from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "jax-gs_amd"))

FIELDS = ("means", "scales", "quaternions", "opacities", "sh_coeffs")
SH_C0 = 0.28209479177387814


def listed():
    """n Gaussians (of which the share `active` is unmasked; 1.0 passes no mask), SH degree
    `degree` in arrays of `coeffs` coefficients, a width x height frame.  `layout` places the
    Gaussians: "box" a uniform box, "clusters" 32 clusters, "dense" most of them in 4 tight
    clusters."""
    def case(name, kind, n, width, height, degree, coeffs, layout="clusters", active=1.0, tpu=False):
        return {"name": name, "kind": kind, "n": n, "width": width, "height": height, "degree": degree,
                "coeffs": coeffs, "layout": layout, "active": active, "tpu": tpu}

    return [
        # a unit-test sized step: latency and launches only
        case("fit_2k_96x64", "fit", 2000, 96, 64, 3, 16),
        # a thumbnail view of a small scene, colour without view dependence
        case("render_16k_256x256", "render", 16384, 256, 256, 0, 1, layout="box"),
        # a camera being refined against a photograph (mean squared error; the background and
        # W2C are differentiated too), odd frame height
        case("pose_50k_640x479", "pose", 50_000, 640, 479, 1, 4),
        # the module functions one after another, as code written against the reference's
        # modules calls them (projection, colours, the full tile arrays, the compositing)
        case("modules_60k_504x378", "modules", 60_000, 504, 378, 2, 9),
        # an object-sized capture at an eighth of the photographs' resolution
        case("fit_200k_504x378", "fit", 200_000, 504, 378, 3, 16),
        # the trainer's own step in the middle of a run: odd frame, padded capacity, SH degree 2 of 3
        case("train_300k_979x546", "train", 300_000, 979, 546, 2, 16, active=0.7),
        # the headline step
        case("fit_1m_1920x1080", "fit", 1_000_000, 1920, 1080, 3, 16),
        # the trainer's step at the headline's size
        case("train_1m_1920x1080", "train", 1_000_000, 1920, 1080, 3, 16),
        # the photometric loss and its gradient on a rendered frame, for programs with a loop of their own
        case("loss_1920x1080", "loss", 0, 1920, 1080, 0, 0),
        # many Gaussians in few tiles: sorting volume, truncated tiles
        case("render_3m_1280x720", "render", 3_000_000, 1280, 720, 1, 4, layout="dense"),
        # padded training capacity with the densification statistics after the backward
        case("stats_2m_1280x720", "stats", 2_097_152, 1280, 720, 3, 16, active=0.6),
        # a 4K view of a large scene through the other rasterizer path
        case("render_2m_3840x2160", "render", 2_000_000, 3840, 2160, 3, 16, tpu=True),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["render", "render", "fit", "fit", "stats", "train", "train", "pose", "modules", "loss"])
    width = _log_uniform(rng, 64, 1920)
    height = max(33, min(1080, int(width * rng.uniform(0.5, 0.85))))
    degree = rng.randrange(4)
    n = _log_uniform(rng, 1500, {"render": 2_000_000, "pose": 400_000, "modules": 200_000}.get(kind, 1_000_000))
    c = {"kind": kind, "n": n, "width": width, "height": height, "degree": degree,
         "coeffs": rng.choice([(degree + 1) ** 2, 16]), "layout": rng.choice(["box", "clusters", "clusters", "dense"]),
         "active": rng.choice([1.0, 0.6, 0.85]), "tpu": rng.random() < 0.3}
    if kind in ("train", "stats"):
        c["coeffs"] = 16
    if kind == "modules":
        c.update(active=1.0, coeffs=(degree + 1) ** 2, tpu=False)
    if kind == "loss":
        c.update(n=0, degree=0, coeffs=0, layout="box", active=1.0, tpu=False)
    return c


# ------------------------------------------------------------------ inputs


def _inputs(case, seed):
    """The seeded inputs as plain tensors on the GPU."""
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev)
    gen.manual_seed(1000003 * seed + 17)
    n, W, H, K = case["n"], case["width"], case["height"], case["coeffs"]

    def rand(*shape):
        return torch.rand(shape, generator=gen, device=dev)

    def randn(*shape):
        return torch.randn(shape, generator=gen, device=dev)

    def spread(lo, hi, *shape):
        return lo + (hi - lo) * rand(*shape)

    x = {}
    if case["kind"] == "loss":
        # a rendered frame and the photograph it is compared with: a smooth picture and noise
        yy = torch.linspace(0, 3.0, H, device=dev)[:, None, None]
        xx = torch.linspace(0, 5.0, W, device=dev)[None, :, None]
        phase = spread(0.0, 6.0, 3)
        photo = 0.5 + 0.3 * torch.sin(xx * 2.0 + phase) * torch.cos(yy * 3.0 - phase) + 0.1 * randn(H, W, 3)
        x["target"] = photo.clamp(0.0, 1.0)
        x["image"] = (photo + 0.05 * randn(H, W, 3)).clamp(0.0, 1.0)
        return x
    focal = (W / 2.0) / math.tan(math.radians(30.0)) if case["layout"] == "box" else 407.0 * W / 504.0
    x["camera"] = (W, H, focal, focal, W / 2.0, H / 2.0)
    w2c = torch.eye(4, device=dev)
    if case["layout"] == "box":
        means = torch.stack([spread(-1, 1, n), spread(-1, 1, n), spread(2, 6, n)], 1)
        size = (-3.5, 0.5)
    elif case["layout"] == "clusters":
        centres = torch.stack([spread(-1.5, 1.5, 32), spread(-1.5, 1.5, 32), spread(1.5, 12.0, 32)], 1)
        which = torch.randint(0, 32, (n,), generator=gen, device=dev)
        means = centres[which] + 0.3 * randn(n, 3)
        size = (-4.0, 0.7)
    else:
        near = int(0.7 * n)
        centres = torch.stack([spread(-0.15, 0.15, 4), spread(-0.1, 0.1, 4), spread(3.5, 4.5, 4)], 1)
        which = torch.randint(0, 4, (near,), generator=gen, device=dev)
        z = spread(2.0, 8.0, n - near)
        far = torch.stack([spread(-1, 1, n - near) * z * (W / 2.0) / focal,
                           spread(-1, 1, n - near) * z * (H / 2.0) / focal, z], 1)
        means = torch.cat([centres[which] + 0.05 * randn(near, 3), far], 0)
        size = (-4.0, 0.7)
    x["means"] = means
    x["scales"] = size[0] + size[1] * randn(n, 3)
    q = randn(n, 4)
    x["quaternions"] = q / q.norm(dim=1, keepdim=True)
    x["opacities"] = randn(n, 1)
    sh = torch.zeros((n, K, 3), device=dev)
    sh[:, 0] = (rand(n, 3) - 0.5) / SH_C0
    used = (case["degree"] + 1) ** 2
    if used > 1:
        sh[:, 1:used] = 0.05 * randn(n, used - 1, 3)
    x["sh_coeffs"] = sh
    x["mask"] = None
    if case["active"] < 1.0 or case["kind"] == "train":
        x["mask"] = rand(n) < case["active"]
        x["opacities"][~x["mask"]] = -20.0
        x["quaternions"][~x["mask"]] = torch.tensor([1.0, 0.0, 0.0, 0.0], device=dev)
    x["background"] = None
    if case["kind"] in ("pose", "modules"):
        x["background"] = rand(3)
    if case["kind"] == "pose":
        # a camera a little off its place: turned by a few hundredths of a radian and moved
        a = 0.03 * randn(3)
        skew = torch.zeros((3, 3), device=dev)
        skew[0, 1], skew[0, 2], skew[1, 2] = -a[2], a[1], -a[0]
        w2c[:3, :3] = torch.linalg.matrix_exp(skew - skew.T)
        w2c[:3, 3] = 0.05 * randn(3)
    x["w2c"] = w2c
    if case["kind"] != "render":
        x["target"] = rand(H, W, 3)
    if case["kind"] == "modules":
        x["cotangent"] = randn(H, W, 3) / (3.0 * H * W)
    if case["kind"] == "train":
        # moments of the size that the gradients of a mean over the frame have
        s = 0.3 / (3.0 * H * W)
        x["mu"] = {f: s * randn(*x[f].shape) for f in FIELDS}
        x["nu"] = {f: s * s * (0.5 + rand(*x[f].shape)) for f in FIELDS}
        x["grad_accum"], x["max_radii"] = 1e-3 * rand(n), torch.floor(20.0 * rand(n))
        x["denom"] = torch.randint(0, 100, (n,), generator=gen, device=dev, dtype=torch.int32)
    if case["kind"] == "stats":
        x["grad_accum"], x["max_radii"] = torch.zeros(n, device=dev), torch.zeros(n, device=dev)
        x["denom"] = torch.zeros(n, device=dev, dtype=torch.int32)
    return x


#: Adam's learning rates at the end of a run, decayed a thousandfold: passes over one state leave the scene as it is.
RATES = {"means": 4.8e-7, "scales": 5e-6, "quaternions": 1e-6, "opacities": 5e-5, "sh_coeffs": 2.5e-6}
STEP_COUNT = 7000


def prepare(case, seed):
    from jax_gs_amd import Camera, Gaussians
    from jax_gs_amd.training.density import DensityState
    from jax_gs_amd.training.optimizer import Adam, AdamState

    x = _inputs(case, seed)
    s = {"case": case}
    if case["kind"] == "loss":
        s["image"], s["target"] = x["image"].requires_grad_(True), x["target"]
        return s
    W, H, fx, fy, cx, cy = x["camera"]
    s["gaussians"] = Gaussians(*[x[f] for f in FIELDS])
    s["camera"] = Camera(W, H, fx, fy, cx, cy, x["w2c"], torch.eye(4, device="cuda:0"))
    for k in ("mask", "background", "target", "cotangent", "w2c"):
        s[k] = x.get(k)
    if case["kind"] == "train":
        s["optimizer"] = Adam(RATES)
        s["state"] = DensityState(s["gaussians"], AdamState(x["mu"], x["nu"], STEP_COUNT),
                                  x["mask"].to(torch.uint8), int(x["mask"].sum()), x["grad_accum"], x["denom"],
                                  x["max_radii"])
    if case["kind"] == "stats":
        s["accum"] = {k: x[k] for k in ("grad_accum", "denom", "max_radii")}
    if case["kind"] not in ("render", "train"):
        s["leaves"] = [x[f].requires_grad_(True) for f in FIELDS]
    if case["kind"] == "pose":
        s["leaves"] += [x["w2c"].requires_grad_(True), x["background"].requires_grad_(True)]
    if case["kind"] == "modules":
        s["leaves"] += [x["background"].requires_grad_(True)]
    return s


# ------------------------------------------------------------------ one pass


def _grads(s):
    return [t.grad for t in s["leaves"]]


def run(s):
    from jax_gs_amd import render, render_l1
    from jax_gs_amd.renderer.projection import project_gaussians
    from jax_gs_amd.renderer.rasterizer import get_tile_interactions, render_tiles
    from jax_gs_amd.renderer.sh import eval_sh
    from jax_gs_amd.training.losses import l1_ssim_loss, mse_loss
    from jax_gs_amd.training.trainer import accumulate_from_extras, train_step

    case = s["case"]
    kind, degree, tpu = case["kind"], case["degree"], case["tpu"]
    if kind == "loss":
        s["image"].grad = None
        total, l1, d_ssim = l1_ssim_loss(s["image"], s["target"])
        total.backward()
        return {"total": total.detach(), "l1": l1.detach(), "d_ssim": d_ssim.detach(), "grad": s["image"].grad}
    g, cam, mask = s["gaussians"], s["camera"], s["mask"]
    if kind == "render":
        with torch.no_grad():
            image, extras = render(g, cam, fast_tpu_rasterizer=tpu, mask=mask, sh_degree=degree)
        return {"image": image, "extras": extras}
    if kind == "train":
        state = s["state"]
        _, loss, metrics = train_step(state, s["target"], s["w2c"], (cam.W, cam.H, cam.fx, cam.fy, cam.cx, cam.cy),
                                      s["optimizer"], fast_tpu_rasterizer=tpu, sh_degree=degree)
        return {"loss": loss, "metrics": metrics, "params": [getattr(g, f) for f in FIELDS],
                "mu": [state.opt_state.mu[f] for f in FIELDS], "nu": [state.opt_state.nu[f] for f in FIELDS],
                "grad_accum": state.grad_accum, "denom": state.denom, "max_radii": state.max_radii}
    for t in s["leaves"]:
        t.grad = None
    if kind == "pose":
        image, extras = render(g, cam, background=s["background"], fast_tpu_rasterizer=tpu, mask=mask,
                               sh_degree=degree)
        loss = mse_loss(image, s["target"])
        loss.backward()
        return {"image": image.detach(), "loss": loss.detach(), "grads": _grads(s), "extras": extras}
    if kind == "modules":
        means2d, cov2d, radii, valid, depths = project_gaussians(g, cam)
        dirs = torch.nn.functional.normalize(g.means, dim=1)  # the camera centre is the origin
        colors = (eval_sh(degree, g.sh_coeffs, dirs) + 0.5).clamp(0.0, 1.0)
        tiles, gids, count = get_tile_interactions(means2d.detach(), radii, valid, depths.detach(), cam.H, cam.W)
        image = render_tiles(means2d, cov2d, g.opacities, colors, tiles, gids, cam.H, cam.W,
                             background=s["background"])
        image.backward(s["cotangent"])
        return {"image": image.detach(), "grads": _grads(s), "tiles": tiles, "gids": gids, "count": count}
    image, loss, extras = render_l1(g, cam, s["target"], fast_tpu_rasterizer=tpu, mask=mask, sh_degree=degree)
    loss.backward()
    out = {"image": image.detach(), "loss": loss.detach(), "grads": _grads(s), "extras": extras}
    if kind == "stats":
        accumulate_from_extras(s["accum"], g.means.grad, g.means.detach(), cam, extras, active=mask)
        out["accum"] = s["accum"]
    return out


# ------------------------------------------------------------------ what a pass cannot do without

#: entries that a pixel blends until it is opaque, and operations of one blend (exponent, quadratic form,
#: weight, three colours) and of its derivative
BLENDS, FORWARD, BACKWARD = 40, 30, 60


def work(case):
    n, K, used = case["n"], case["coeffs"], (case["degree"] + 1) ** 2
    pixels = case["width"] * case["height"]
    if case["kind"] == "loss":
        # two images read, one gradient written; two separable 11-tap blurs of five and three planes
        return {"bytes": 36.0 * pixels, "flops": 3.0 * pixels * 8 * 2 * 22}
    read = n * (44 + 12 * used) + (n if case["active"] < 1.0 else 0)  # parameters, mask
    image = 12.0 * pixels
    blends = pixels * min(BLENDS, n)
    if case["kind"] == "render":
        return {"bytes": read + 5.0 * n + image, "flops": float(FORWARD * blends)}
    flops = float((FORWARD + BACKWARD) * blends)
    grads = n * (44 + 12 * K)
    if case["kind"] == "train":
        # parameters and two moments read and written, the statistics likewise
        return {"bytes": 6.0 * grads + 24.0 * n + image, "flops": flops + 3.0 * pixels * 8 * 2 * 22}
    if case["kind"] == "modules":
        return {"bytes": read + grads + 2048.0 * n + 2 * image, "flops": flops}
    return {"bytes": read + 5.0 * n + grads + 2 * image + (36.0 * n if case["kind"] == "stats" else 0), "flops": flops}


def tolerance(case):
    """32-bit arithmetic throughout: four times the error against ``exact`` that was measured (images 8e-7, gradients
    9e-6, the loss's gradient 7e-7).  A pixel whose transmittance lies at the threshold may take one more entry
    (1e-4 of its colour).  The derivative of an L1 mean is the sign of each value's difference, which turns where an
    image meets its target to within rounding: a few values of a frame, each with the step of its cotangent."""
    if case["kind"] == "loss":
        return {"rel": 1e-5, "max": 1e-3}
    if case["kind"] in ("fit", "stats", "train"):
        return {"rel": min(0.03, 2.0 * math.sqrt(4.0 / (3 * case["width"] * case["height"]))), "max": 0.9}
    return {"rel": 4e-5, "max": 2e-2}


# ------------------------------------------------------------------ the same in 64 bits


def _sh_basis(degree, d):
    x, y, z = d[:, 0], d[:, 1], d[:, 2]
    b = [torch.full_like(x, SH_C0)]
    if degree > 0:
        b += [-0.4886025119029199 * y, 0.4886025119029199 * z, -0.4886025119029199 * x]
    if degree > 1:
        b += [1.0925484305920792 * x * y, -1.0925484305920792 * y * z,
              0.31539156525252005 * (2 * z * z - x * x - y * y), -1.0925484305920792 * x * z,
              0.5462742152960396 * (x * x - y * y)]
    if degree > 2:
        b += [-0.5900435899266435 * y * (3 * x * x - y * y), 2.890611442640554 * x * y * z,
              -0.4570457994644658 * y * (4 * z * z - x * x - y * y),
              0.3731763325901154 * z * (2 * z * z - 3 * x * x - 3 * y * y),
              -0.4570457994644658 * x * (4 * z * z - x * x - y * y), 1.445305721320277 * z * (x * x - y * y),
              -0.5900435899266435 * x * (x * x - 3 * y * y)]
    return torch.stack(b, 1)


def _project(case, camera, p, w2c, mask):
    """Per Gaussian: centre, conic, opacity and colour of its splat (one array of nine), radius, validity, depth."""
    _, _, fx, fy, cx, cy = camera
    cam = p["means"] @ w2c[:3, :3].T + w2c[:3, 3]
    x, y, z = cam.unbind(1)
    r, i, j, k = (p["quaternions"] / p["quaternions"].norm(dim=1, keepdim=True)).unbind(1)
    rot = torch.stack([1 - 2 * (j * j + k * k), 2 * (i * j - r * k), 2 * (i * k + r * j),
                       2 * (i * j + r * k), 1 - 2 * (i * i + k * k), 2 * (j * k - r * i),
                       2 * (i * k - r * j), 2 * (j * k + r * i), 1 - 2 * (i * i + j * j)], 1).view(-1, 3, 3)
    m = rot * torch.exp(p["scales"])[:, None, :]
    sigma = m @ m.transpose(1, 2).contiguous()
    zs = z.clamp(min=0.01)
    zero = torch.zeros_like(z)
    jac = torch.stack([fx / zs, zero, -fx * x / zs ** 2, zero, fy / zs, -fy * y / zs ** 2], 1).view(-1, 2, 3)
    jw = jac @ w2c[:3, :3].contiguous()
    cov = jw @ sigma @ jw.transpose(1, 2).contiguous()
    a, b, c = cov[:, 0, 0] + 0.3, cov[:, 0, 1], cov[:, 1, 1] + 0.3
    det = a * c - b * b
    radius = torch.ceil(3 * torch.sqrt((a + c) / 2 + torch.sqrt((((a + c) / 2) ** 2 - det).clamp(min=0))))
    det = det.clamp(min=1e-6)
    centre = -(w2c[:3, :3].T @ w2c[:3, 3])
    view = p["means"] - centre
    basis = _sh_basis(case["degree"], view / view.norm(dim=1, keepdim=True))
    used = basis.shape[1]
    colour = ((basis[:, :, None] * p["sh_coeffs"][:, :used]).sum(1) + 0.5).clamp(0, 1)
    valid = z > 0.01
    if mask is not None:
        valid = valid & mask
    splat = torch.cat([(fx * x / z + cx)[:, None], (fy * y / z + cy)[:, None], (c / det)[:, None], (-b / det)[:, None],
                       (a / det)[:, None], torch.sigmoid(p["opacities"]), colour], 1)
    return splat, radius, valid, z


def _entries(camera, splat, radius, valid, z):
    """The (tile, Gaussian) entries in the rasterizer's order: tile, the depth's leading 13 bits, Gaussian."""
    W, H = camera[:2]
    tx, ty = (W + 15) // 16, (H + 15) // 16
    mx, my = splat[:, 0], splat[:, 1]
    on = valid & (mx + radius > 0) & (mx - radius < W) & (my + radius > 0) & (my - radius < H)
    ids = on.nonzero()[:, 0]
    mx, my, radius = mx[ids], my[ids], radius[ids]

    def span(m, size):
        lo = torch.div((m - radius).clamp(0, size - 1), 16, rounding_mode="floor").long()
        hi = torch.div((m + radius).clamp(0, size - 1), 16, rounding_mode="floor").long()
        return lo, torch.minimum(hi - lo + 1, torch.full_like(lo, 16))

    x0, nx = span(mx, W)
    y0, ny = span(my, H)
    quantum = z[ids].float().view(torch.int32).long() >> 18
    of = torch.repeat_interleave(torch.arange(ids.numel(), device=ids.device), nx * ny)
    k = torch.arange(of.numel(), device=ids.device) - (torch.cumsum(nx * ny, 0) - nx * ny)[of]
    tile = (y0[of] + k // nx[of]) * tx + x0[of] + k % nx[of]
    _, order = torch.sort((tile << 13) | quantum[of], stable=True)
    gids = ids[of[order]]
    start = torch.searchsorted(tile[order].contiguous(), torch.arange(tx * ty + 1, device=ids.device))
    return gids, start


def _blend(camera, splat, gids, start, tiles, background):
    """The pixels [tiles, 256, 3] of some tiles."""
    W = camera[0]
    tx = (W + 15) // 16
    dev = splat.device
    lane = torch.arange(256, device=dev)
    px = (tiles % tx * 16)[:, None] + lane % 16 + 0.5
    py = (torch.div(tiles, tx, rounding_mode="floor") * 16)[:, None] + torch.div(lane, 16, rounding_mode="floor") + 0.5
    count = (start[tiles + 1] - start[tiles]).clamp(max=4096)
    T = torch.ones_like(px, dtype=torch.float64)
    C = torch.zeros((tiles.numel(), 256, 3), dtype=torch.float64, device=dev)
    live = (count > 0).nonzero()[:, 0]
    k = 0
    while live.numel():
        at = k + torch.arange(64, device=dev)
        there = at[None] < count[live][:, None]
        g = gids[(start[tiles[live]][:, None] + at).clamp(max=gids.numel() - 1)]
        e = splat[g]  # [live, 64, 9]
        dx = px[live][:, None, :] - e[:, :, 0, None]
        dy = py[live][:, None, :] - e[:, :, 1, None]
        power = -0.5 * (dx * dx * e[:, :, 2, None] + 2 * dx * dy * e[:, :, 3, None] + dy * dy * e[:, :, 4, None])
        seen = (power > -10.0) & there[:, :, None]
        alpha = torch.where(seen, torch.exp(power) * e[:, :, 5, None], torch.zeros_like(power)).clamp(max=0.99)
        passed = torch.cumsum(torch.log1p(-alpha), 1)
        before = T[live][:, None] * torch.exp(passed - torch.log1p(-alpha))
        alpha = alpha * (before > 1e-4)
        C = C.index_add(0, live, (alpha * before).transpose(1, 2).contiguous() @ e[:, :, 6:].contiguous())
        T = T.index_copy(0, live, T[live] * torch.exp(torch.log1p(-alpha).sum(1)))
        k += 64
        live = live[(count[live] > k) & (T[live] > 1e-4).any(1)]
    return C + T[:, :, None] * background


def _frame(camera, tiles, pixels):
    """[tiles, 256, 3] <-> [H, W, 3]: the tiles' pixels that lie in the frame."""
    W, H = camera[:2]
    tx, ty = (W + 15) // 16, (H + 15) // 16
    return pixels.view(ty, tx, 16, 16, 3).permute(0, 2, 1, 3, 4).reshape(ty * 16, tx * 16, 3)[:H, :W]


def _unframe(camera, image):
    W, H = camera[:2]
    tx, ty = (W + 15) // 16, (H + 15) // 16
    full = image.new_zeros((ty * 16, tx * 16, 3))
    full[:H, :W] = image
    return full.view(ty, 16, tx, 16, 3).permute(0, 2, 1, 3, 4).reshape(ty * tx, 256, 3)


def _photometric(image, target, lam=0.2):
    """((1 - lam) L1 + lam D-SSIM, L1, D-SSIM)."""
    x = torch.arange(11, device=image.device, dtype=torch.float64) - 5
    w = torch.exp(-x * x / (2 * 1.5 ** 2))
    w = w / w.sum()

    def blur(t):
        t = torch.nn.functional.pad(t, (0, 0, 5, 5, 5, 5))
        t = sum(w[k] * t[k:k + image.shape[0]] for k in range(11))
        return sum(w[k] * t[:, k:k + image.shape[1]] for k in range(11))

    m1, m2 = blur(image), blur(target)
    s11 = (blur(image * image) - m1 * m1).clamp(min=0)
    s22 = (blur(target * target) - m2 * m2).clamp(min=0)
    s12 = blur(image * target) - m1 * m2
    c1, c2 = 0.01 ** 2, 0.03 ** 2
    ssim = ((2 * m1 * m2 + c1) * (2 * s12 + c2) / ((m1 * m1 + m2 * m2 + c1) * (s11 + s22 + c2))).clamp(-1, 1).mean()
    l1 = (image - target).abs().mean()
    d = ((1 - ssim) / 2).clamp(min=0)
    return (1 - lam) * l1 + lam * d, l1, d


def exact(case, seed):
    kind = case["kind"]
    x = _inputs(case, seed)
    if kind == "loss":
        image = x["image"].double().requires_grad_(True)
        total, l1, d = _photometric(image, x["target"].double())
        total.backward()
        return {"total": total.detach(), "l1": l1.detach(), "d_ssim": d.detach(), "grad": image.grad}
    cam = x["camera"]
    W, H = cam[:2]
    p = {f: x[f].double().requires_grad_(kind != "render") for f in FIELDS}
    w2c = x["w2c"].double().requires_grad_(kind == "pose")
    bg = (torch.zeros(3, device="cuda:0") if x["background"] is None else x["background"]).double()
    bg.requires_grad_(kind in ("pose", "modules"))
    with torch.set_grad_enabled(kind != "render"):
        splat, radius, valid, z = _project(case, cam, p, w2c, x["mask"])
    leaf = splat.detach().requires_grad_(True)
    with torch.no_grad():
        gids, start = _entries(cam, splat.detach(), radius, valid, z)
        every = torch.arange(start.numel() - 1, device=gids.device)
        pixels = torch.cat([_blend(cam, leaf, gids, start, part, bg) for part in every.split(2048)])
        image = _frame(cam, every, pixels)
    out = {"image": image, "extras": None}
    if kind == "render":
        return out
    shown = image.clone().requires_grad_(True)
    target = x["target"].double()
    if kind == "modules":
        cot = x["cotangent"].double()
    else:
        if kind == "train":
            loss, l1, d = _photometric(shown, target)
        elif kind == "pose":
            loss = ((shown - target) ** 2).mean()
        else:
            loss = (shown - target).abs().mean()
        loss.backward()
        cot, loss = shown.grad, loss.detach()
    cot = _unframe(cam, cot)
    for part in every.split(512):
        (_blend(cam, leaf, gids, start, part, bg) * cot[part]).sum().backward()
    splat.backward(leaf.grad)
    grads = [p[f].grad for f in FIELDS]
    if kind == "modules":
        return {"image": image, "grads": grads + [bg.grad], "tiles": None, "gids": None, "count": None}
    out.update(loss=loss, grads=grads + ([w2c.grad, bg.grad] if kind == "pose" else []))
    if kind in ("train", "stats"):
        depth = z.detach().clamp(min=0.01)
        accum = x["grad_accum"].double() + grads[0].norm(dim=1) * depth / ((cam[2] + cam[3]) / 2) * (W * H * 3.0)
        if kind == "stats":
            out["accum"] = {"grad_accum": accum, "denom": None, "max_radii": None}
            return out
        mu = {f: 0.1 * g + 0.9 * x["mu"][f].double() for f, g in zip(FIELDS, grads)}
        nu = {f: 0.001 * g * g + 0.999 * x["nu"][f].double() for f, g in zip(FIELDS, grads)}
        new = []
        for f in FIELDS:
            t = STEP_COUNT + 1
            step = RATES[f] * (mu[f] / (1 - 0.9 ** t)) / (torch.sqrt(nu[f] / (1 - 0.999 ** t)) + 1e-8)
            rows = x["mask"].view(-1, *[1] * (step.dim() - 1))
            new.append(x[f].double() - step * rows)
        return {"loss": loss, "metrics": {"l1": l1.detach(), "ssim": (1 - 2 * d).detach()}, "params": new,
                "mu": [mu[f] for f in FIELDS], "nu": [nu[f] for f in FIELDS], "grad_accum": accum, "denom": None,
                "max_radii": None}
    return out
