"""GPU parity: rasterize / rasterize_backward vs the CPU oracle.

Tolerances (north star): image max abs error <= 1e-4 on the [0,1] scale,
gradients relative L2 <= 1e-3.  On the reference's constant fixtures the
reference's own thresholds apply (scripts/check_cuda_gradients.py:610-616,
771-777: rendered rel <= 1e-6, points/conic rel <= 2e-3, opacity/colour rel
<= 1e-5); they are met here with margin.
"""

from __future__ import annotations

import pytest
import torch

import helpers
import cuda_rasterizer as cr
from oracle import blend, preprocess
from oracle import render as orender

pytestmark = pytest.mark.gpu

INPUTS = ("points_image", "cov_inv_image", "opacities", "colors")


@pytest.fixture(params=[1, 2, 4])
def waves(request):
    """The blend kernels run each tile on 1, 2 or 4 waves (gs_set_blend_waves)."""
    cr.set_blend_waves(request.param)
    yield request.param
    cr.set_blend_waves(0)


def _thresholds(f):
    return (f["width"], f["height"], f["tile_size"], f["alpha_threshold"],
            f["transmittance_threshold"], f["chi_squared_threshold"])


@pytest.mark.parametrize("name", ["multitile", "truncated"])
def test_reference_fixtures(gpu, name, waves):
    f = helpers.fixture_tensors(name)
    off, ids = cr.compute_tile_intersection(f["points_image"].to(gpu), f["radii"].to(gpu),
                                            f["depths"].to(gpu), f["mask"].to(gpu), f["width"],
                                            f["height"], f["tile_size"])
    assert off.cpu().tolist() == f["expected_indexing_offset"]
    args = _thresholds(f)
    ins = [f[k].clone().requires_grad_(True) for k in INPUTS]
    ref = blend.rasterize_bruteforce(off.cpu(), ids.cpu(), *ins, *args)
    (ref * f["upstream"]).sum().backward()
    image = cr.rasterize(off, ids, *[f[k].to(gpu) for k in INPUTS], *args)
    assert helpers.rel_l2(image, ref) <= 1e-6
    assert helpers.max_abs(image, ref) <= 1e-6
    grads = cr.rasterize_backward(f["upstream"].to(gpu), off, ids, *[f[k].to(gpu) for k in INPUTS],
                                  *args)
    limits = [2e-4, 2e-4, 1e-5, 1e-5]  # points, conic, opacity, colour
    for nm, a, t, lim in zip(INPUTS, grads, ins, limits):
        assert helpers.rel_l2(a, t.grad) <= lim, nm
        assert helpers.cosine(a, t.grad) >= 0.99999, nm


def _shared_inputs(scene, sh_sigmoid=False):
    """Projection, colours and layout from the oracle (CPU), used as identical
    inputs by both rasterizers."""
    p, cam, target = scene
    scales, quats, opac = helpers.activated(p)
    out = orender.render_stages(cam["w2c"], cam["K"], cam["width"], cam["height"], p["means"],
                                scales, quats, opac, p["sh_dc"], p["sh_rest"], sh_sigmoid=sh_sigmoid)
    keep = out["proj"]["keep"]
    k2 = keep.unsqueeze(1)
    z = torch.zeros_like(opac)
    leaves = dict(points_image=torch.where(k2, out["points_image"], 0.0).detach(),
                  cov_inv_image=torch.where(k2, out["conic"], 0.0).detach(),
                  opacities=torch.where(keep, opac, z).detach(),
                  colors=out["colors"].detach())
    return leaves, out["indexing_offset"], out["gaussian_ids_sorted"], cam, target


SCENES = {
    "cfg1": lambda: helpers.scene_box(10_000, 256, 256, 300.0, seed=0),
    "cfg2cam_small": lambda: helpers.scene_orbit(20_000, 320, 240, 440.0, seed=5),
    "large_splats": lambda: helpers.scene_box(1_500, 100, 70, 80.0, seed=6, log_scale=(-1.8, 0.5),
                                              z=(1.0, 5.0)),
}


@pytest.fixture(params=[0, 1 << 62])
def four_arrays(request, monkeypatch):
    """The gradients summed in rows and copied, or in the four arrays, whatever the lists."""
    monkeypatch.setattr(cr, "_FOUR_ARRAYS_KEYS", request.param)


@pytest.mark.parametrize("name", list(SCENES))
def test_gradient_routes(gpu, name, four_arrays):
    """Every seed of the backward by either route: the oracle's gradients (as
    test_rasterize_shared_inputs), and for display and L1 the sums of the other entries."""
    leaves, off, ids, cam, target = _shared_inputs(SCENES[name]())
    W, H = cam["width"], cam["height"]
    args = (W, H, 16, 1e-4, 1e-4, 9.21)
    ins = [leaves[k].clone().requires_grad_(True) for k in INPUTS]
    ref = blend.rasterize(off, ids, *ins, *args)
    up = torch.randn(H, W, 3, generator=torch.Generator().manual_seed(9))
    (ref.clamp(0, 1) * 255 * up).sum().backward()
    d = [off.to(gpu), ids.to(gpu)] + [leaves[k].to(gpu) for k in INPUTS]
    image = cr.rasterize(*d, *args)
    inner = ((image >= 0) & (image <= 1)).float() * 255  # the clamp's gradient
    up = up.to(gpu)
    for got in (cr.rasterize_backward(up * inner, *d, *args, rendered_image=image),
                cr.rasterize_display_backward(up, *d, *args, rendered_image=image)):
        for nm, a, t in zip(INPUTS, got, ins):
            assert a.is_contiguous() and helpers.rel_l2(a, t.grad) <= 1e-3, nm
    one = torch.ones(1, device=gpu)
    l1 = cr.rasterize_l1_backward(target.to(gpu), one, *d, W, H, image, 1e-4, 1e-4, 9.21)
    rows = cr.rasterize_l1_backward_rows(target.to(gpu), one, *d, W, H, image, 1e-4, 1e-4, 9.21)
    for nm, a, b in zip(INPUTS, l1, (rows[:, :2], rows[:, 2:5], rows[:, 5], rows[:, 6:])):
        assert a.is_contiguous() and helpers.rel_l2(a, b) <= 1e-5, nm


@pytest.mark.parametrize("name", list(SCENES))
def test_rasterize_shared_inputs(gpu, name, waves):
    leaves, off, ids, cam, target = _shared_inputs(SCENES[name]())
    W, H = cam["width"], cam["height"]
    args = (W, H, 16, 1e-4, 1e-4, 9.21)
    ins = [leaves[k].clone().requires_grad_(True) for k in INPUTS]
    ref = blend.rasterize(off, ids, *ins, *args)
    up = torch.randn(H, W, 3, generator=torch.Generator().manual_seed(9))
    (ref * up).sum().backward()
    d = [leaves[k].to(gpu) for k in INPUTS]
    image = cr.rasterize(off.to(gpu), ids.to(gpu), *d, *args)
    assert helpers.max_abs(image.clamp(0, 1), ref.clamp(0, 1)) <= 1e-4
    assert helpers.rel_l2(image, ref) <= 1e-5
    g_saved = cr.rasterize_backward(up.to(gpu), off.to(gpu), ids.to(gpu), *d, *args,
                                    rendered_image=image)
    g_replay = cr.rasterize_backward(up.to(gpu), off.to(gpu), ids.to(gpu), *d, *args)
    for nm, a, b, t in zip(INPUTS, g_saved, g_replay, ins):
        assert helpers.rel_l2(a, t.grad) <= 1e-3, nm
        assert helpers.rel_l2(b, a) <= 1e-5, nm


@pytest.mark.parametrize("tile", [8, 32])
def test_rasterize_generic_tile_sizes(gpu, tile):
    p, cam, _ = helpers.scene_box(3_000, 96, 72, 100.0, seed=8, log_scale=(-3.0, 0.5))
    scales, quats, opac = helpers.activated(p)
    pts, depths, _, conic, radii, mask = preprocess.project_points(
        p["means"], scales, quats, opac, cam["w2c"], cam["K"], 0.01, 100.0, 1 / 255, 0.5, 128.0, 96, 72)
    colors = torch.rand(3_000, 3, generator=torch.Generator().manual_seed(1))
    opac_m = torch.where(mask, opac, torch.zeros_like(opac))
    d = lambda t: t.detach().to(gpu)  # noqa: E731
    off, ids = cr.compute_tile_intersection(d(pts), d(radii), d(depths), d(mask), 96, 72, tile)
    args = (96, 72, tile, 1e-4, 1e-4, 9.21)
    ins = [t.detach().clone().requires_grad_(True) for t in (pts, conic, opac_m, colors)]
    ref = blend.rasterize(off.cpu(), ids.cpu(), *ins, *args)
    up = torch.randn(72, 96, 3, generator=torch.Generator().manual_seed(2))
    (ref * up).sum().backward()
    image = cr.rasterize(off, ids, *[d(t) for t in ins], *args)
    assert helpers.max_abs(image.clamp(0, 1), ref.clamp(0, 1)) <= 1e-4
    grads = cr.rasterize_backward(up.to(gpu), off, ids, *[d(t) for t in ins], *args)
    for a, t in zip(grads, ins):
        assert helpers.rel_l2(a, t.grad) <= 1e-3


@pytest.mark.parametrize("alpha_thr,chi,t_thr", [(0.0, 9.21, 1e-4), (1e-4, 9.21, 1e-4),
                                                 (0.05, 9.21, 1e-4), (1e-4, 4.0, 1e-4),
                                                 (-0.05, 9.21, 0.0)])
def test_rasterize_thresholds_and_opacity_extremes(gpu, alpha_thr, chi, t_thr, waves):
    """The 16x16 kernels' inclusion test (E below min(chi, 2 ln(o / alpha_thr)), staged
    per record) against the oracle's separate chi-square and alpha tests, with
    zero, tiny, near-one and negative opacities among the Gaussians and several
    thresholds: image <= 1e-4, gradients relative L2 <= 1e-3.  A negative
    opacity gives alpha = o exp(-E/2) < 0: skipped (zero gradient) for
    alpha_thr >= 0, composited where alpha >= alpha_thr < 0 (there with
    transmittance threshold 0: T can then grow, and the oracle's zeroing of
    T < T_thr differs from stopping the pixel)."""
    p, cam, _ = helpers.scene_box(3_000, 96, 72, 100.0, seed=12, log_scale=(-3.0, 0.5))
    scales, quats, opac = helpers.activated(p)
    pts, depths, _, conic, radii, mask = preprocess.project_points(
        p["means"], scales, quats, opac, cam["w2c"], cam["K"], 0.01, 100.0, 0.0, 0.5, 128.0, 96, 72)
    opac = opac.detach().clone()
    opac[::7] = 0.0
    opac[1::7] = 1e-6
    opac[2::7] = 0.9999
    opac[3::7] = -0.3 * opac[3::7]
    colors = torch.rand(3_000, 3, generator=torch.Generator().manual_seed(3))
    opac_m = torch.where(mask, opac, torch.zeros_like(opac))
    d = lambda t: t.detach().to(gpu)  # noqa: E731
    off, ids = cr.compute_tile_intersection(d(pts), d(radii), d(depths), d(mask), 96, 72, 16)
    args = (96, 72, 16, alpha_thr, t_thr, chi)
    ins = [t.detach().clone().requires_grad_(True) for t in (pts, conic, opac_m, colors)]
    ref = blend.rasterize(off.cpu(), ids.cpu(), *ins, *args)
    up = torch.randn(72, 96, 3, generator=torch.Generator().manual_seed(4))
    (ref * up).sum().backward()
    image = cr.rasterize(off, ids, *[d(t) for t in ins], *args)
    assert helpers.max_abs(image.clamp(0, 1), ref.clamp(0, 1)) <= 1e-4
    grads = cr.rasterize_backward(up.to(gpu), off, ids, *[d(t) for t in ins], *args,
                                  rendered_image=image)
    for a, t in zip(grads, ins):
        assert helpers.rel_l2(a, t.grad) <= 1e-3


def test_rasterize_edge_cases(gpu):
    W, H = 40, 24
    off = torch.zeros(6, dtype=torch.int32, device=gpu)
    ids = torch.zeros(0, dtype=torch.int32, device=gpu)
    z = lambda *s: torch.zeros(*s, device=gpu)  # noqa: E731
    image = cr.rasterize(off, ids, z(3, 2), z(3, 3), z(3), z(3, 3), W, H, 16, 1e-4, 1e-4, 9.21)
    assert image.shape == (H, W, 3) and float(image.abs().max()) == 0.0
    grads = cr.rasterize_backward(torch.ones(H, W, 3, device=gpu), off, ids, z(3, 2), z(3, 3), z(3),
                                  z(3, 3), W, H, 16, 1e-4, 1e-4, 9.21)
    assert all(float(g.abs().max()) == 0.0 for g in grads)
    # transmittance threshold above 1: nothing is composited
    f = helpers.fixture_tensors("multitile")
    offs = torch.tensor(f["expected_indexing_offset"], dtype=torch.int32, device=gpu)
    idss = torch.tensor(f["expected_gaussian_ids_sorted"], dtype=torch.int32, device=gpu)
    image = cr.rasterize(offs, idss, *[f[k].to(gpu) for k in INPUTS], 48, 48, 16, 0.0, 2.0, 9.21)
    assert float(image.abs().max()) == 0.0
    # out-of-range ids are ignored instead of read
    bad = idss.clone()
    bad[0] = 10_000
    image = cr.rasterize(offs, bad, *[f[k].to(gpu) for k in INPUTS], 48, 48, 16, 0.0, 0.0, 9.21)
    assert torch.isfinite(image).all()


def _ptr(t):
    return t.data_ptr() if t is not None else None


def test_backward_overwrite_and_accumulate_modes(gpu):
    """gs_rasterize_backward through the C ABI: accumulate=0 overwrites whatever the
    outputs held; accumulate=1 adds to it."""
    from cuda_rasterizer import _lib

    leaves, off, ids, cam, _ = _shared_inputs(SCENES["cfg2cam_small"]())
    W, H = cam["width"], cam["height"]
    d = [leaves[k].to(gpu) for k in INPUTS]
    off, ids = off.to(gpu), ids.to(gpu)
    up = torch.randn(H, W, 3, generator=torch.Generator().manual_seed(3)).to(gpu)
    want = cr.rasterize_backward(up, off, ids, *d, W, H, 16, 1e-4, 1e-4, 9.21)
    n = d[0].shape[0]
    shapes = [(n, 2), (n, 3), (n,), (n, 3)]
    stream = torch.cuda.current_stream(gpu).cuda_stream
    for mode, fill in ((0, float("nan")), (1, 1.5)):
        outs = [torch.full(s, fill, device=gpu) for s in shapes]
        st = _lib.load().gs_rasterize_backward(
            _ptr(up), None, _ptr(off), _ptr(ids), off.numel(), ids.numel(), *[_ptr(t) for t in d],
            n, W, H, 16, 1e-4, 1e-4, 9.21, *[_ptr(t) for t in outs], mode, stream)
        assert st == 0
        torch.cuda.synchronize()
        for nm, got, ref in zip(INPUTS, outs, want):
            expect = ref if mode == 0 else ref + 1.5
            assert helpers.rel_l2(got, expect) <= 1e-5, (mode, nm)


def _work_counts(off, ids, pts, conic, opac, W, H, ts, a_thr, t_thr, chi):
    """Reference blend loop trip counts (src/cuda/kernel.cu:954-982), numpy per tile."""
    import numpy as np

    off, ids = off.cpu().numpy(), ids.cpu().numpy()
    pts, conic, opac = (t.detach().cpu().numpy().astype(np.float32) for t in (pts, conic, opac))
    tx = (W + ts - 1) // ts
    visited = composited = 0
    ends = np.append(off[1:], len(ids))
    for t in range(len(off)):
        g = ids[off[t]:ends[t]]
        if len(g) == 0:
            continue
        x0, y0 = (t % tx) * ts, (t // tx) * ts
        ys, xs = np.mgrid[y0:min(y0 + ts, H), x0:min(x0 + ts, W)]
        du = xs.ravel()[None, :].astype(np.float32) - pts[g, 0:1]
        dv = ys.ravel()[None, :].astype(np.float32) - pts[g, 1:2]
        A, B, C = conic[g, 0:1], conic[g, 1:2], conic[g, 2:3]
        E = A * du * du + np.float32(2) * B * du * dv + C * dv * dv
        alpha = np.exp(np.float32(-0.5) * E) * opac[g, None]
        inc = (E < chi) & (alpha >= a_thr)
        T = np.cumprod(np.where(inc, (1 - alpha) + np.float32(1e-10), 1), axis=0)
        stop = inc & (T < t_thr)
        has = stop.any(axis=0)
        first = np.where(has, stop.argmax(axis=0), len(g) - 1)
        visited += int((first + 1).sum())
        rows = np.arange(len(g))[:, None]
        composited += int((inc & (rows <= first[None, :])).sum())
    return visited, composited


def test_rasterize_work_counts(gpu):
    leaves, off, ids, cam, _ = _shared_inputs(SCENES["cfg2cam_small"]())
    W, H = cam["width"], cam["height"]
    v_ref, c_ref = _work_counts(off, ids, leaves["points_image"], leaves["cov_inv_image"],
                                leaves["opacities"], W, H, 16, 1e-4, 1e-4, 9.21)
    v, c = cr.rasterize_work(off.to(gpu), ids.to(gpu), leaves["points_image"].to(gpu),
                             leaves["cov_inv_image"].to(gpu), leaves["opacities"].to(gpu), W, H,
                             16, 1e-4, 1e-4, 9.21)
    assert v_ref > 0 and c_ref > 0
    # exp implementations differ in the last bits: an entry at the alpha threshold may flip
    assert abs(v - v_ref) <= 1e-4 * v_ref and abs(c - c_ref) <= 1e-4 * c_ref


@pytest.mark.parametrize("opaque,t_thr", [(False, 1e-4), (True, 1e-4), (False, 0.0)])
@pytest.mark.parametrize("count", [1, 3, 4, 5, 8, 63, 65, 130])
def test_backward_pending_entries(gpu, waves, count, opaque, t_thr):
    """The backward reduces four entries at a time: list lengths around multiples of
    four and of a batch, also with pixels that an opacity of exactly 1 saturates
    (alpha 1 at the splat's centre) and with no transmittance threshold.  The sums run
    in float32 in another order than the oracle's: about sqrt(256) roundings of 6e-8
    on terms of either sign, 1e-5 of the result here."""
    W, H = 19, 17  # 2 x 2 tiles, three of them partial
    g = torch.Generator().manual_seed(count)
    pts = torch.rand(count, 2, generator=g) * torch.tensor([W - 1.0, H - 1.0])
    if opaque:
        pts = pts.round()
    scale = torch.rand(count, generator=g) * 0.2 + 0.02
    conic = torch.stack([scale, 0.3 * scale, 1.5 * scale], dim=1)
    opac = torch.rand(count, generator=g) * 0.8 + 0.1
    if opaque:
        opac[count // 2] = 1.0
    col = torch.rand(count, 3, generator=g)
    ids = torch.arange(count, dtype=torch.int32).repeat(4)
    off = torch.arange(4, dtype=torch.int32) * count
    args = (W, H, 16, 1e-4, t_thr, 9.21)
    ins = [t.clone().requires_grad_(True) for t in (pts, conic, opac, col)]
    image = blend.rasterize(off, ids, *ins, *args)
    up = torch.randn(H, W, 3, generator=g)
    (image * up).sum().backward()
    d = [t.to(gpu) for t in (pts, conic, opac, col)]
    img = cr.rasterize(off.to(gpu), ids.to(gpu), *d, *args)
    assert helpers.max_abs(img, image) <= 1e-5
    got = cr.rasterize_backward(up.to(gpu), off.to(gpu), ids.to(gpu), *d, *args,
                                rendered_image=img)
    for nm, a, t in zip(INPUTS, got, ins):
        assert a.is_contiguous() and helpers.rel_l2(a, t.grad) <= 1e-4, nm
    # the rows and the four arrays of the L1 seed hold the same sums (atomics in any order)
    target, one = torch.rand(H, W, 3, generator=g).to(gpu), torch.ones(1, device=gpu)
    l1 = (target, one, off.to(gpu), ids.to(gpu), *d, W, H, img, 1e-4, t_thr, 9.21)
    want = cr.rasterize_l1_backward(*l1, accumulators=torch.zeros(9 * count, device=gpu))
    rows = cr.rasterize_l1_backward_rows(*l1)
    for nm, a, b in zip(INPUTS, want, (rows[:, :2], rows[:, 2:5], rows[:, 5], rows[:, 6:])):
        assert helpers.rel_l2(b, a) <= 1e-5, nm


def _one_tile_images(gpu, pts, conic, opac, col, t_thr):
    """One 16x16 tile with every entry in index order, composited by 1, 2 and 4 waves."""
    n = pts.shape[0]
    d = [t.to(gpu) for t in (pts, conic, opac, col)]
    off = torch.zeros(1, dtype=torch.int32, device=gpu)
    ids = torch.arange(n, dtype=torch.int32, device=gpu)
    out = []
    for w in (1, 2, 4):
        cr.set_blend_waves(w)
        out.append(cr.rasterize(off, ids, *d, 16, 16, 16, 1e-4, t_thr, 9.21).cpu())
    cr.set_blend_waves(0)
    return out


@pytest.mark.parametrize("bad", ["colour", "opacity"])
def test_batches_after_a_special_one(gpu, bad):
    """A batch with a non-finite colour or opacity is composited with selects and leaves
    finished pixels with 0 < T < the threshold; the ordinary batches that follow (lists of
    three batches of the widest form, whose first two leave the right columns open) add
    nothing to them.  Equal bits for every wave count, and the oracle's image beyond the
    special splat's reach (1e-5: about 20 products of rounded factors)."""
    n, g = 768, torch.Generator().manual_seed(5)
    pts = torch.rand(n, 2, generator=g) * 16
    pts[:512, 0] *= 6 / 16
    conic = torch.tensor([[0.2, 0.0, 0.2]]).repeat(n, 1)  # a reach of 6.8 pixels
    opac = torch.rand(n, generator=g) * 0.2 + 0.1
    col = torch.rand(n, 3, generator=g)
    pts[3], conic[3] = torch.tensor([2.0, 2.0]), torch.tensor([4.0, 0.0, 4.0])  # 1.5 pixels
    plain = [pts, conic, opac.clone(), col.clone()]
    if bad == "colour":
        col[3, 1] = float("nan")
    else:
        opac[3] = float("nan")
    images = _one_tile_images(gpu, pts, conic, opac, col, 0.5)
    for image in images[1:]:
        assert helpers.same(image, images[0])
    plain[2][3] = 0.0
    ref = blend.rasterize(torch.zeros(1, dtype=torch.int32), torch.arange(n, dtype=torch.int32),
                          *plain, 16, 16, 16, 1e-4, 0.5, 9.21)
    far = torch.ones(16, 16, dtype=torch.bool)
    far[:5, :5] = False
    assert helpers.max_abs(images[0][far], ref[far]) <= 1e-5


def test_finished_pixels_and_an_unbounded_alpha(gpu):
    """A conic that is not positive definite gives alpha = exp2(900): infinite where it is
    composited, and nothing to the pixels that opaque splats finished before."""
    n = 40
    pts = torch.tensor([[2.0, 8.0]]).repeat(n, 1)
    conic = torch.tensor([[0.05, 0.0, 0.001]]).repeat(n, 1)  # columns 0..15, E = 8.5 at the last
    opac, col = torch.full((n,), 0.99), torch.rand(n, 3, generator=torch.Generator().manual_seed(6))
    conic[6:, 0] = 1.0  # six reach the whole tile and finish its columns 0..4
    pts[20], conic[20] = torch.tensor([60.0, 8.0]), torch.tensor([-1.0, 0.0, 1.0])
    images = _one_tile_images(gpu, pts, conic, opac, col, 1e-4)
    for image in images[1:]:
        assert helpers.same(image, images[0])
    keep = torch.arange(n) != 20
    ref = blend.rasterize(torch.zeros(1, dtype=torch.int32),
                          torch.arange(n - 1, dtype=torch.int32), pts[keep], conic[keep],
                          opac[keep], col[keep], 16, 16, 16, 1e-4, 1e-4, 9.21)
    assert helpers.max_abs(images[0][:, :5], ref[:, :5]) <= 1e-5
    assert not torch.isfinite(images[0][:, 15]).any()  # composited there


@pytest.mark.parametrize("t_thr", [1e-30, 1e-10, 0.0])
def test_backward_small_thresholds(gpu, waves, t_thr):
    """Pixels composited down to T of 1e-29 with gradients of 1e18: what the sums leave of
    1e18 by rounding (1e11) over T would be infinite, and infinity times a weight of 0 NaN.
    Relative 1e-4: the sums' roundings, sqrt(256) of 6e-8 on terms of either sign."""
    n, g = 70, torch.Generator().manual_seed(7)
    pts = torch.rand(n, 2, generator=g) * 4 + 6
    conic = torch.tensor([[0.05, 0.0, 0.05]]).repeat(n, 1)
    opac, col = torch.full((n,), 0.9), torch.rand(n, 3, generator=g)
    off, ids = torch.zeros(1, dtype=torch.int32), torch.arange(n, dtype=torch.int32)
    args = (16, 16, 16, 1e-4, t_thr, 9.21)
    ins = [t.clone().requires_grad_(True) for t in (pts, conic, opac, col)]
    up = torch.randn(16, 16, 3, generator=g)
    (blend.rasterize(off, ids, *ins, *args) * up).sum().backward()
    d = [t.to(gpu) for t in (pts, conic, opac, col)]
    off, ids = off.to(gpu), ids.to(gpu)
    image = cr.rasterize(off, ids, *d, *args)
    got = cr.rasterize_backward(1e18 * up.to(gpu), off, ids, *d, *args, rendered_image=image)
    for nm, a, t in zip(INPUTS, got, ins):
        assert helpers.rel_l2(a / 1e18, t.grad) <= 1e-4, nm
