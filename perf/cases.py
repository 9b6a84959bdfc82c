"""What a user of this rasterizer has it do, as cases that can be timed and checked.

Each case is one call sequence of a user's program:
  step      a training step of the library loop: render_l1 (optionally with the SSIM term and
            the densification statistics), then backward
  captured  the same step replayed from a HIP graph (CapturedStep)
  loop      a training step of the reference-shaped loop: PyTorch activations, render(),
            L1 and fused_ssim on the image, backward
  seven     the same loop around the seven extension functions, as a program that keeps its
            own wrapper composes them (render_unfused)
  view      a rendered image without gradients: a viewer, an evaluation
  bin       compute_tile_intersection alone
  ssim      fused_ssim forward and backward
  adam      one optimizer step over all parameters

Scenes: "box" (10k-type scene in front of the camera), "ball" (an object seen from an orbit)
and "cluster" (50 clusters in a wide uniform cloud, a share of them `large` splats).
"""

from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "3dgs_from_scratch_amd"))

import cuda_rasterizer as cr  # noqa: E402
from cuda_rasterizer.fused import render_l1  # noqa: E402
from cuda_rasterizer.graphs import CapturedStep  # noqa: E402
from cuda_rasterizer.train import DEFAULT_LR, Densifier, FusedAdam  # noqa: E402
from cuda_rasterizer.wrapper import render, render_unfused  # noqa: E402

NAMES = ("means", "log_scales", "quats_raw", "opacity_logits", "sh_dc", "sh_rest")
RENDERS = ("step", "captured", "loop", "seven", "view")
NEAR, FAR, MIN_OPACITY, MIN_RADIUS, MAX_RADIUS = 0.01, 100.0, 1 / 255, 0.5, 128.0
ALPHA, TRANSMITTANCE, CHI = 1e-4, 1e-4, 9.21


def _case(name, path, scene="ball", n=0, width=0, height=0, sh=3, ssim=0.0, large=0.0,
          densify=False, batch=1, hwc=True, padding="valid"):
    c = dict(path=path, scene=scene, n=n, width=width, height=height, sh=sh, ssim=ssim,
             large=large, densify=densify, batch=batch, hwc=hwc, padding=padding)
    return dict(c, name=name) if name else c


def listed():
    return [
        # a small scene's preview in a viewer, an odd window size: latency
        _case("view_20k_251x183", "view", "box", 20_000, 251, 183),
        # the smallest training step: a toy scene with constant colours
        _case("step_10k_256x256", "step", "box", 10_000, 256, 256, sh=0),
        # a small object's step replayed from a graph, camera and target copied in
        _case("captured_100k_800x800", "captured", "ball", 100_000, 800, 800),
        # an early training step with the full loss and the densification statistics
        _case("step_200k_1280x720_ssim", "step", "ball", 200_000, 1280, 720, ssim=0.2,
              densify=True),
        # the benchmark's training step: a full scene at 1080p
        _case("step_1m_1920x1080", "step", "cluster", 1_000_000, 1920, 1080),
        # training at 4K with a grown scene: the largest image and lists
        _case("step_2m_3840x2160", "step", "cluster", 2_000_000, 3840, 2160),
        # the reference's training loop on photographs of an odd size, full loss
        _case("loop_300k_979x547_ssim", "loop", "ball", 300_000, 979, 547, ssim=0.2),
        # a program with its own wrapper around the seven functions, larger odd photographs
        _case("seven_600k_1599x1063", "seven", "cluster", 600_000, 1599, 1063),
        # an evaluation render of a large scene with many large splats
        _case("view_3m_1920x1080_large", "view", "cluster", 3_000_000, 1920, 1080, large=0.05),
        # the tile lists alone, for a program that blends by itself
        _case("bin_1m_2560x1440", "bin", "cluster", 1_000_000, 2560, 1440),
        # SSIM as a loss on two planar images of an odd size
        _case("ssim_2x3x1063x1599", "ssim", batch=2, width=1599, height=1063, hwc=False,
              padding="same"),
        # one optimizer step of a full scene
        _case("adam_1m", "adam", "cluster", 1_000_000),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """Paths, scenes and options as listed, sizes over the logarithm of the range."""
    path = rng.choice(("step", "step", "captured", "loop", "seven", "view", "view", "bin",
                       "ssim", "adam"))
    scene = rng.choice(("box", "ball", "cluster"))
    n = _log(rng, 5_000, 120_000 if scene == "box" else 1_000_000)
    width = _log(rng, 200, 2560)
    height = min(max(150, int(width * rng.uniform(0.5, 1.0))), 4_200_000 // width)
    if path == "ssim":
        return _case(None, path, batch=rng.randint(1, 2), width=width, height=height,
                     hwc=rng.random() < 0.5, padding=rng.choice(("same", "valid")))
    if path == "adam":
        return _case(None, path, scene, n)
    if path == "captured":  # what a graph is for: steps that the host would bound
        n, width, height = min(n, 300_000), min(width, 1280), min(height, 1280)
    lam = rng.choice((0.0, 0.2)) if path in ("step", "loop", "captured") else 0.0
    return _case(None, path, scene, n, width, height, sh=rng.choice((0, 3, 3)), ssim=lam,
                 large=rng.choice((0.0, 0.0, 0.05)) if scene == "cluster" else 0.0,
                 densify=path == "step" and rng.random() < 0.5)


# ---------------------------------------------------------------- inputs


def _look_at(azimuth, elevation, dist):
    """World-to-camera of an OpenCV camera on a sphere around the origin, looking at it."""
    c = torch.tensor([dist * math.cos(elevation) * math.cos(azimuth), dist * math.sin(elevation),
                      dist * math.cos(elevation) * math.sin(azimuth)], dtype=torch.float64)
    f = -c / c.norm()
    right = torch.linalg.cross(f, torch.tensor([0.0, -1.0, 0.0], dtype=torch.float64))
    right = right / right.norm()
    rows = torch.stack([right, torch.linalg.cross(f, right), f])
    m = torch.eye(4, dtype=torch.float64)
    m[:3, :3] = rows
    m[:3, 3] = -rows @ c
    return m.float()


def _inputs(case, seed):
    """(parameters, world_to_camera, intrinsic, target) on the GPU, from the seed alone."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(int(seed))
    n, width, height = case["n"], max(case["width"], 1), max(case["height"], 1)

    def rand(*s):
        return torch.rand(*s, generator=g, device=dev)

    def randn(*s):
        return torch.randn(*s, generator=g, device=dev)

    w2c = torch.eye(4)
    if case["scene"] == "box":  # in front of the camera
        means = torch.cat([rand(n, 2) * 2 - 1, rand(n, 1) * 4 + 2], dim=1)
        focal, scale, spread, opacity = 300 / 256, -4.0, 0.5, 1.0
    elif case["scene"] == "ball":  # an object of radius 1.5 from an orbit of radius 4
        d = randn(n, 3)
        means = d / d.norm(dim=1, keepdim=True) * 1.5 * rand(n, 1) ** (1 / 3)
        focal, scale, spread, opacity = 1100 / 800, -4.5, 0.6, 1.5
        if width > height:
            focal = 1000 / 1280
        az, el = rand(2).tolist()
        w2c = _look_at(az * 2 * math.pi, (el * 2 - 1) * math.pi / 3, 4.0)
    else:  # 70% around 50 centres in view, 30% uniform around the camera
        k = int(round(0.7 * n))
        cz = rand(50) * 8 + 2
        cx, cy = (rand(50) * 1.2 - 0.6) * cz, (rand(50) * 0.7 - 0.35) * cz
        which = torch.randint(0, 50, (k,), generator=g, device=dev)
        means = torch.cat([torch.stack([cx, cy, cz], 1)[which] + randn(k, 3) * 0.3,
                           rand(n - k, 3) * 20 - 10])
        focal, scale, spread, opacity = 1400 / 1920, -3.5, 0.8, 1.5
    log_scales = randn(n, 3) * spread + scale
    if case["large"] > 0:
        big = (rand(n) < case["large"]).unsqueeze(1)
        log_scales = torch.where(big, randn(n, 3) * 0.3 - 1.0, log_scales)
    params = dict(means=means.contiguous(), log_scales=log_scales, quats_raw=randn(n, 4),
                  opacity_logits=randn(n) * opacity, sh_dc=randn(n, 3) * 0.3,
                  sh_rest=randn(n, 15, 3) * 0.05 if case["sh"] else torch.zeros(n, 15, 3, device=dev))
    f = focal * width
    intrinsic = torch.tensor([[f, 0.0, width / 2], [0.0, f, height / 2], [0.0, 0.0, 1.0]])
    return params, w2c.to(dev), intrinsic.to(dev), rand(height, width, 3)


def _images(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    shape = (case["batch"], case["height"], case["width"], 3)
    y = torch.rand(*shape, generator=g, device="cuda")
    x = (y + 0.1 * torch.randn(*shape, generator=g, device="cuda")).clamp(0, 1)
    x, y = x.permute(0, 3, 1, 2), y.permute(0, 3, 1, 2)
    return (x, y) if case["hwc"] else (x.contiguous(), y.contiguous())


def _near(case):
    return 0.2 if case["scene"] == "cluster" else NEAR


def _activated(p):
    return (torch.exp(p["log_scales"]),
            p["quats_raw"] / torch.norm(p["quats_raw"], dim=1, keepdim=True).clamp_min(1e-12),
            torch.sigmoid(p["opacity_logits"]))


def _adam_state(case, seed):
    """Parameters, gradients and moments of a training run under way."""
    p = _inputs(case, seed)[0]
    g = torch.Generator(device="cuda").manual_seed(int(seed) + 1_000_003)

    def like(t, s):
        return torch.randn(t.shape, generator=g, device=t.device) * s

    return (p, {k: like(t, 1e-4) for k, t in p.items()}, {k: like(t, 1e-5) for k, t in p.items()},
            {k: like(t, 1e-5) ** 2 for k, t in p.items()})


def prepare(case, seed):
    s = dict(case=dict(case))
    if case["path"] == "ssim":
        s["img"], s["target"] = _images(case, seed)
        s["img"].requires_grad_(True)
        return s
    if case["path"] == "adam":
        p, grads, m, v = _adam_state(case, seed)
        opt = FusedAdam({k: t.requires_grad_(True) for k, t in p.items()},
                        means_decay_steps=30_000)
        for k in p:
            p[k].grad = grads[k]
            opt.exp_avg[k].copy_(m[k])
            opt.exp_avg_sq[k].copy_(v[k])
            opt.step_count[k] = 100
        return dict(s, opt=opt)
    if case["path"] == "bin":
        # one scene's splats in an order drawn from the seed: lists of other Gaussians and
        # ties, and as many entries for every seed
        p, w2c, K, _ = _inputs(case, 7)
        g = torch.Generator(device=w2c.device).manual_seed(int(seed))
        rows = torch.randperm(case["n"], generator=g, device=w2c.device)
        scales, quats, opac = (t[rows] for t in _activated(p))
        pts, depths, _, _, radii, mask = cr.project_points(
            p["means"][rows], scales, quats, opac, w2c, K, _near(case), FAR, MIN_OPACITY,
            MIN_RADIUS, MAX_RADIUS, case["width"], case["height"])
        return dict(s, splats=(pts, radii, depths, mask))
    p, w2c, K, target = _inputs(case, seed)
    s.update(w2c=w2c, K=K, target=target)
    if case["path"] == "view":  # a viewer activates its scene once
        s["scene"] = (p["means"], *_activated(p), p["sh_dc"], p["sh_rest"])
        return s
    s["leaves"] = {k: t.requires_grad_(True) for k, t in p.items()}
    if case["densify"]:
        s["densifier"] = Densifier(case["n"], w2c.device)
    if case["path"] == "captured":
        s["camera"], s["photo"] = w2c.clone(), target.clone()  # what each replay copies in

        def step():
            loss, display, _, _ = _render_l1(s)
            return (loss.detach(), display) + torch.autograd.grad(loss, list(s["leaves"].values()))

        s["graph"] = CapturedStep(step)
    return s


# ---------------------------------------------------------------- one pass


def _render_l1(s):
    c, p = s["case"], s["leaves"]
    return render_l1(s["w2c"], s["K"], c["width"], c["height"], *(p[k] for k in NAMES),
                     s["target"], near_plane=_near(c), densifier=s.get("densifier"),
                     ssim_lambda=c["ssim"])


def _out(loss, display, grads, densifier=None):
    out = dict(loss=loss.detach(), display=display.detach(), grads=dict(zip(NAMES, grads)))
    if densifier is not None:
        out["densify"] = dict(grads=densifier.grads, count=densifier.count)
    return out


def run(s):
    c = s["case"]
    path = c["path"]
    if path == "step":
        for t in s["leaves"].values():
            t.grad = None
        loss, display, _, _ = _render_l1(s)
        loss.backward()
        return _out(loss, display, [s["leaves"][k].grad for k in NAMES], s.get("densifier"))
    if path == "captured":
        s["w2c"].copy_(s["camera"])
        s["target"].copy_(s["photo"])
        s["graph"].replay()
        loss, display, *grads = s["graph"].output
        return _out(loss, display, grads)
    if path in ("loop", "seven"):
        p = s["leaves"]
        for t in p.values():
            t.grad = None
        scales, quats, opac = _activated(p)
        display, _, _ = (render if path == "loop" else render_unfused)(
            s["w2c"], s["K"], c["width"], c["height"], p["means"], scales, quats, opac,
            p["sh_dc"], p["sh_rest"], near_plane=_near(c))
        norm = display / 255.0
        loss = torch.nn.functional.l1_loss(norm, s["target"])
        if c["ssim"] > 0:
            ssim = cr.fused_ssim(norm.permute(2, 0, 1).unsqueeze(0),
                                 s["target"].permute(2, 0, 1).unsqueeze(0), padding="valid")
            loss = (1 - c["ssim"]) * loss + c["ssim"] * (1.0 - ssim)
        loss.backward()
        return _out(loss, display, [p[k].grad for k in NAMES])
    if path == "view":
        with torch.no_grad():
            display, points, radii = render(s["w2c"], s["K"], c["width"], c["height"],
                                            *s["scene"], near_plane=_near(c))
        return dict(display=display, points=points, radii=radii)
    if path == "bin":
        offset, ids = cr.compute_tile_intersection(*s["splats"], c["width"], c["height"])
        return dict(offset=offset, ids=ids)
    if path == "ssim":
        s["img"].grad = None
        mean = cr.fused_ssim(s["img"], s["target"], padding=c["padding"])
        mean.backward()
        return dict(mean=mean.detach(), grad=s["img"].grad)
    s["opt"].step()
    opt = s["opt"]
    return dict(params={k: t.detach() for k, t in opt.params.items()}, m=opt.exp_avg,
                v=opt.exp_avg_sq)


# ---------------------------------------------------------------- cost and tolerance

PARAM_FLOATS = 59  # means 3, log_scales 3, quats 4, opacity 1, SH 48


def _visited(case):
    """Estimated (entry, pixel) pairs that the compositing evaluates: splats over a pixel, until
    the pixel is opaque.  From the mean splat area (E < chi is an ellipse of area pi * chi *
    sigma_u * sigma_v) and the share of the image that the scene covers."""
    n, width, height = case["n"], case["width"], case["height"]
    if case["scene"] == "cluster":
        f, z, seen, cover, spread, scale, stop = 1400 / 1920 * width, 6.0, 0.65, 1.0, 0.8, -3.5, 130
    elif case["scene"] == "ball":
        f = (1000 / 1280 if width > height else 1100 / 800) * width
        z, seen, spread, scale, stop = 4.0, 1.0, 0.6, -4.5, 90
        cover = min(1.0, math.pi * (1.5 * f / z) ** 2 / (width * height))
    else:
        f, z, seen, spread, scale, stop = 300 / 256 * width, 4.0, 0.9, 0.5, -4.0, 90
        cover = min(1.0, (2 * f / z) ** 2 / (width * height))
    sigma2 = (math.exp(scale) * f / z) ** 2 * math.exp(spread ** 2) + 0.3
    depth = n * seen * math.pi * CHI * sigma2 / (width * height * cover)
    return min(depth, stop) * cover * width * height


def work(case):
    pixels = case["width"] * case["height"]
    if case["path"] == "ssim":
        values = 3 * case["batch"] * pixels
        # both images read, the gradient written; 5 statistics forward and 3 maps back, each
        # filtered by 11 + 11 taps, and about 60 operations of their arithmetic
        return dict(bytes=12 * values, flops=values * ((5 + 3) * 2 * 22 + 60))
    n = case["n"]
    if case["path"] == "adam":  # p, g, m, v read; p, m, v written
        return dict(bytes=7 * 4 * PARAM_FLOATS * n, flops=12 * PARAM_FLOATS * n)
    keys = _visited(case) / 12.0  # listed (tile, Gaussian) entries, long lists cut by opacity
    if case["path"] == "bin":  # points, radii, depths, mask read; the lists written
        return dict(bytes=21 * n + 4 * keys, flops=20 * n)
    pairs = _visited(case)
    scene = 4 * PARAM_FLOATS * n
    if case["path"] == "view":
        return dict(bytes=scene + 16 * n + 12 * pixels, flops=22 * pairs + 300 * n)
    ssim = 3 * pixels * ((5 + 3) * 2 * 22 + 60) if case["ssim"] else 0
    return dict(bytes=2 * scene + 24 * pixels, flops=92 * pairs + 900 * n + ssim)


def tolerance(case):
    if case["path"] == "bin":
        return "exact"
    if case["path"] == "adam":  # 4e-8 from 64 bits
        return dict(rel=2e-7, max=1e-5)
    if case["path"] == "ssim":  # 7e-7 from 64 bits
        return dict(rel=4e-6, max=1e-3)
    if case["path"] == "view":  # 3e-7 to 1.6e-5 from 64 bits: pixels at an edge of a splat
        return dict(rel=5e-5, max=0.05)
    # gradients: sums by atomics in any order (up to 7e-5 from run to run), and pixels whose
    # rounding takes them over an edge of a splat or of the loss (3e-5 to 8e-4 from 64 bits over
    # the listed cases, a few Gaussians off by more)
    return dict(rel=2e-3, max=0.5)


# ---------------------------------------------------------------- the same in 64 bits

SH_1 = 0.4886025119029199
SH_2 = (1.0925484305920792, 0.31539156525252005, 0.5462742152960396)
SH_3 = (0.5900435899266435, 2.890611442640554, 0.4570457994644658, 0.3731763325901154,
        1.445305721320277)


def _colours64(p, w2c):
    cam = -w2c[:3, :3].t() @ w2c[:3, 3]
    d = p["means"] - cam
    x, y, z = (d / d.norm(dim=1, keepdim=True)).unbind(1)
    xx, yy, zz = x * x, y * y, z * z
    basis = torch.stack([
        -SH_1 * y, SH_1 * z, -SH_1 * x,
        SH_2[0] * x * y, SH_2[0] * y * z, SH_2[1] * (3 * zz - 1), SH_2[0] * x * z,
        SH_2[2] * (xx - yy),
        SH_3[0] * y * (xx - yy), SH_3[1] * x * y * z, SH_3[2] * y * (4 * zz - xx - yy),
        SH_3[3] * z * (2 * zz - 3 * xx - 3 * yy), SH_3[2] * x * (4 * zz - xx - yy),
        SH_3[4] * z * (xx - yy), SH_3[0] * x * (xx - 3 * yy)], dim=1)
    raw = p["sh_dc"] * 0.28209479177387814 + (p["sh_rest"] * basis.unsqueeze(-1)).sum(1)
    return torch.clamp_min(raw + 0.5, 0.0)


def _project64(p, w2c, K, width, height, near):
    """(points, radii, conic, opacity, keep), differentiable."""
    scales, quats, opac = _activated(p)
    cam = p["means"] @ w2c[:3, :3].t() + w2c[:3, 3]
    xc, yc, zc = cam.unbind(1)
    fx, fy, cx, cy = K[0, 0], K[1, 1], K[0, 2], K[1, 2]
    zc = torch.where(zc > near, zc, torch.ones_like(zc))
    u, v = fx * xc / zc + cx, fy * yc / zc + cy
    qx, qy, qz, qw = quats.unbind(1)
    rot = torch.stack([
        1 - 2 * (qy * qy + qz * qz), 2 * (qx * qy - qz * qw), 2 * (qx * qz + qy * qw),
        2 * (qx * qy + qz * qw), 1 - 2 * (qx * qx + qz * qz), 2 * (qy * qz - qx * qw),
        2 * (qx * qz - qy * qw), 2 * (qy * qz + qx * qw), 1 - 2 * (qx * qx + qy * qy)],
        dim=1).reshape(-1, 3, 3)
    xn, yn = xc / zc, yc / zc
    lx, ly = 1.3 * max(cx, width - cx) / fx, 1.3 * max(cy, height - cy) / fy
    xn = torch.where(xn.abs() <= lx, xn, xn.clamp(-lx, lx).detach())
    yn = torch.where(yn.abs() <= ly, yn, yn.clamp(-ly, ly).detach())
    zero = torch.zeros_like(zc)
    jac = torch.stack([fx / zc, zero, -fx * xn / zc, zero, fy / zc, -fy * yn / zc],
                      dim=1).reshape(-1, 2, 3)
    t = (jac.unsqueeze(-1) * w2c[:3, :3]).sum(2)  # (N, 2, 3)
    m = (t.unsqueeze(-1) * rot.unsqueeze(1)).sum(2) * scales.unsqueeze(1)
    a, b, c = (m[:, 0] ** 2).sum(1) + 0.3, (m[:, 0] * m[:, 1]).sum(1), (m[:, 1] ** 2).sum(1) + 0.3
    det = torch.clamp_min(a * c - b * b, 1e-12)
    ru, rv = 3 * torch.sqrt(a), 3 * torch.sqrt(c)
    with torch.no_grad():
        z = cam[:, 2]
        r = torch.maximum(ru, rv)
        keep = ((opac >= MIN_OPACITY) & (z > near) & (z < FAR) & (r >= MIN_RADIUS)
                & (r <= MAX_RADIUS) & (u > -ru) & (u < width + ru) & (v > -rv) & (v < height + rv))
    return (torch.stack([u, v], 1), torch.stack([ru, rv], 1).detach(),
            torch.stack([c / det, -b / det, a / det], 1), opac, keep)


def _lists64(points, radii, depth, keep, width, height):
    """(start, length, ids) of each 16x16 tile's entries in (depth, index) order."""
    rows = torch.nonzero(keep).squeeze(1)
    rows = rows[torch.sort(depth[rows], stable=True).indices]
    p, r = points[rows], radii[rows]
    lo = torch.floor(p - r)
    hi = torch.floor(p + r)
    most = torch.tensor([width - 1, height - 1], device=p.device, dtype=p.dtype)
    lo, hi = (torch.minimum(t.clamp_min(0), most).long() // 16 for t in (lo, hi))
    span = hi - lo + 1
    count = span[:, 0] * span[:, 1]
    at = torch.repeat_interleave(torch.arange(rows.numel(), device=p.device), count)
    local = torch.arange(at.numel(), device=p.device) - (count.cumsum(0) - count)[at]
    tiles_x, tiles_y = (width + 15) // 16, (height + 15) // 16
    tile = (lo[at, 1] + local // span[at, 0]) * tiles_x + lo[at, 0] + local % span[at, 0]
    tile, order = torch.sort(tile.int(), stable=True)
    length = torch.bincount(tile, minlength=tiles_x * tiles_y)
    return length.cumsum(0) - length, length, rows[at[order]].int()


def _entries64(splat, tile, tiles_x, through):
    """alpha (tiles, entries, 256) and the share of light before each entry.  splat: (tiles,
    entries, 9) with u, v, conic, opacity, colour; through: light that reaches the first."""
    px = torch.arange(256, device=tile.device)
    pu = ((tile % tiles_x * 16).unsqueeze(1) + px % 16).double().unsqueeze(1)
    pv = ((tile // tiles_x * 16).unsqueeze(1) + px // 16).double().unsqueeze(1)
    f = [splat[..., k].unsqueeze(-1) for k in range(6)]
    du, dv = pu - f[0], pv - f[1]
    e = f[2] * du * du + 2 * f[3] * du * dv + f[4] * dv * dv
    alpha = torch.where(e < CHI, torch.exp(-0.5 * e) * f[5], torch.zeros_like(e))
    alpha = torch.where(alpha >= ALPHA, alpha, torch.zeros_like(alpha))
    t = torch.cumprod(torch.cat([through.unsqueeze(1), 1 - alpha + 1e-10], dim=1), dim=1)
    before = torch.where(t[:, :-1] >= TRANSMITTANCE, t[:, :-1], torch.zeros_like(alpha))
    return alpha, before, t[:, -1]


def _blend64(splats, start, length, ids, width, height, grad_of=None):
    """The image (H, W, 3); with grad_of (image -> its gradient), also the splats' gradients."""
    dev = splats.device
    tiles_x, tiles_y = (width + 15) // 16, (height + 15) // 16
    n_tiles = tiles_x * tiles_y
    light = torch.ones(n_tiles, 256, dtype=torch.float64, device=dev)
    image = torch.zeros(n_tiles, 256, 3, dtype=torch.float64, device=dev)
    used = torch.zeros_like(length)
    none = torch.cat([splats, torch.zeros_like(splats[:1])])  # a last row that adds nothing

    def gather(tile, first, count):
        k = first + torch.arange(count, device=dev)
        at = start[tile].unsqueeze(1) + k
        row = ids[at.clamp_max(max(ids.numel() - 1, 0))].long()
        return torch.where(k < length[tile].unsqueeze(1), row, splats.shape[0])

    live = torch.nonzero(length > 0).squeeze(1)
    first, step = 0, 64
    while live.numel():
        for part in live.split(1024):
            splat = none[gather(part, first, step)]
            alpha, before, after = _entries64(splat, part, tiles_x, light[part])
            image[part] += (alpha * before).transpose(1, 2) @ splat[..., 6:]
            light[part] = after
        first += step
        used[live] = first
        live = live[(light[live].amax(1) >= TRANSMITTANCE) & (length[live] > first)]
    used = torch.minimum(used, length)

    def frame(t):
        t = t.reshape(tiles_y, tiles_x, 16, 16, 3).permute(0, 2, 1, 3, 4)
        return t.reshape(tiles_y * 16, tiles_x * 16, 3)[:height, :width]

    whole = frame(image)
    if grad_of is None:
        return whole, None
    g = torch.nn.functional.pad(grad_of(whole), (0, 0, 0, tiles_x * 16 - width, 0,
                                                 tiles_y * 16 - height))
    g = g.reshape(tiles_y, 16, tiles_x, 16, 3).permute(0, 2, 1, 3, 4).reshape(n_tiles, 256, 3)
    total = torch.zeros_like(none)
    order = torch.sort(used, descending=True, stable=True).indices
    at, most = 0, 1 << 24
    counts = used[order].tolist()
    while at < n_tiles and counts[at] > 0:
        take = max(1, most // (256 * counts[at]))
        part = order[at:at + take]
        rows = gather(part, 0, counts[at])
        splat = none[rows].requires_grad_(True)
        one = torch.ones(part.numel(), 256, dtype=torch.float64, device=dev)
        with torch.enable_grad():
            alpha, before, _ = _entries64(splat, part, tiles_x, one)
            ((alpha * before).transpose(1, 2) @ splat[..., 6:]).backward(g[part])
        total.index_add_(0, rows.reshape(-1), splat.grad.reshape(-1, 9))
        at += take
    return whole, total[:-1]


def _ssim64(x, y, padding):
    """Mean SSIM of (B, C, H, W) images: 11-tap Gaussian window, sigma 1.5, zero padding."""
    w = torch.exp(-torch.arange(-5, 6, dtype=torch.float64) ** 2 / 4.5)
    w = (w / w.sum()).tolist()

    def blur(t):
        h, v = t.shape[-2:]
        t = torch.nn.functional.pad(t, (5, 5, 5, 5))
        t = sum(w[k] * t[..., k:k + v] for k in range(11))
        return sum(w[k] * t[..., k:k + h, :] for k in range(11))

    m1, m2 = blur(x), blur(y)
    s1, s2, s12 = blur(x * x) - m1 * m1, blur(y * y) - m2 * m2, blur(x * y) - m1 * m2
    s = ((2 * m1 * m2 + 1e-4) * (2 * s12 + 9e-4)
         / ((m1 * m1 + m2 * m2 + 1e-4) * (s1 + s2 + 9e-4)))
    return (s[..., 5:-5, 5:-5] if padding == "valid" else s).mean()


def exact(case, seed):
    path = case["path"]
    if path == "bin":  # whole numbers
        return None
    if path == "ssim":
        x, y = (t.double() for t in _images(case, seed))
        x.requires_grad_(True)
        mean = _ssim64(x, y, case["padding"])
        return dict(mean=mean.detach(), grad=torch.autograd.grad(mean, x)[0])
    if path == "adam":
        p, g, m, v = ({k: t.double() for k, t in d.items()} for d in _adam_state(case, seed))
        out = dict(params={}, m={}, v={})
        for k in p:
            out["m"][k] = 0.9 * m[k] + 0.1 * g[k]
            out["v"][k] = 0.999 * v[k] + 0.001 * g[k] ** 2
            out["params"][k] = p[k] - DEFAULT_LR[k] * (out["m"][k] / (1 - 0.9 ** 101)) / (
                torch.sqrt(out["v"][k] / (1 - 0.999 ** 101)) + 1e-15)
        return out
    p32, w2c32, K, target = _inputs(case, seed)
    if path != "view" and _visited(case) > 5e9:
        return None
    width, height = case["width"], case["height"]
    # the depth order is one of 32-bit values, ties by index, and a change of it changes the image
    w = w2c32[2]
    m = p32["means"]
    depth = w[0] * m[:, 0] + w[1] * m[:, 1] + w[2] * m[:, 2] + w[3]
    p = {k: t.double().requires_grad_(path != "view") for k, t in p32.items()}
    w2c = w2c32.double()
    points, radii, conic, opac, keep = _project64(p, w2c, K.double(), width,
                                                  height, _near(case))
    with torch.no_grad():
        start, length, ids = _lists64(points, radii, depth, keep, width, height)
    splats = torch.cat([points, conic, opac.unsqueeze(1), _colours64(p, w2c)], dim=1)
    if path == "view":
        image, _ = _blend64(splats, start, length, ids, width, height)
        k = keep.unsqueeze(1)
        return dict(display=image.clamp(0, 1) * 255, points=torch.where(k, points, 0.0),
                    radii=torch.where(k, radii, 0.0))
    seen = {}

    def grad_of(image):
        image = image.detach().requires_grad_(True)
        norm = image.clamp(0, 1)
        loss = (norm - target.double()).abs().mean()
        if case["ssim"] > 0:
            x, y = (t.permute(2, 0, 1).unsqueeze(0) for t in (norm, target.double()))
            loss = (1 - case["ssim"]) * loss + case["ssim"] * (1 - _ssim64(x, y, "valid"))
        seen["loss"], seen["display"] = loss.detach(), norm.detach() * 255
        return torch.autograd.grad(loss, image)[0]

    with torch.no_grad():
        _, g = _blend64(splats.detach(), start, length, ids, width, height,
                        torch.enable_grad()(grad_of))
    grads = torch.autograd.grad(splats, [p[k] for k in NAMES], g)
    out = dict(loss=seen["loss"], display=seen["display"], grads=dict(zip(NAMES, grads)))
    if case["densify"]:
        ndc = g[:, :2] * torch.tensor([width / 2, height / 2], device=g.device)
        out["densify"] = dict(grads=torch.where(keep, ndc.norm(dim=1), 0.0), count=keep.double())
    return out
