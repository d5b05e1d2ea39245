"""GPU parity of the L1 + SSIM image loss (crates/splat-train-loss) against
the CPU oracle on identical inputs.

Bar: bit for bit.  Both sides sum every blur tap, SSIM term and tile total in
one fixed order with unfused f32 arithmetic, so the tile partials, SSIM
coefficients, loss map and dL/dpred agree exactly; the device total of the
partials agrees with their float64 sum to 1e-6.
"""
import numpy as np
import pytest
import torch

import vauss_amd as va
from oracle import pyoracle as po
from tests._util import to_gpu
from vauss_amd import scenes

pytestmark = pytest.mark.gpu

OPTS = [dict(), dict(composite_bg=(0.2, 0.5, 0.9)), dict(mask=True), dict(alpha_weight=0.3),
        dict(composite_bg=(1.0, 0.0, 0.3), mask=True, alpha_weight=0.1)]


def _case(h, w, cn, seed):
    rng = np.random.default_rng(seed)
    gt = rng.integers(0, 1 << 32, (h, w), dtype=np.uint64).astype(np.uint32)
    g = np.stack([(gt >> (8 * k)) & 0xFF for k in range(4)], -1).astype(np.float32) / 255.0
    pred = (0.7 * g[..., :cn] + 0.3 * rng.uniform(0, 1, (h, w, cn))).astype(np.float32)
    return pred, gt


def _cfgs(opts, l1_w=0.8, ssim_w=-0.2):
    cfg = va.ImageLossConfig(l1_w, ssim_w, opts.get("composite_bg"), opts.get("mask", False),
                             opts.get("alpha_weight", 0.0))
    ocfg = po.loss_cfg(l1_w, ssim_w, opts.get("alpha_weight", 0.0), opts.get("composite_bg"), opts.get("mask", False))
    return cfg, ocfg


def _check(pred, gt, opts, dl_kind):
    cfg, ocfg = _cfgs(opts)
    h, w, cn = pred.shape
    print(f"[case] {h}x{w}x{cn} {opts} dl={dl_kind}", flush=True)
    pd = torch.from_numpy(pred).cuda()
    gd = torch.from_numpy(gt.view(np.int32)).cuda()
    partials, coeffs, total = va.image_loss_forward_train(pd, gd, cfg)
    lmap = va.image_loss_eval(pd, gd, cfg)
    rp, rc, rm = po.image_loss_forward(pred, gt, ocfg)
    np.testing.assert_array_equal(partials.cpu().numpy().view(np.uint32), rp.view(np.uint32))
    np.testing.assert_array_equal(coeffs.cpu().numpy().view(np.uint32), rc.view(np.uint32))
    np.testing.assert_array_equal(lmap.cpu().numpy().view(np.uint32), rm.view(np.uint32))
    want_total = rp.astype(np.float64).sum()
    assert abs(float(total.item()) - want_total) <= 1e-6 * abs(want_total) + 1e-9
    if dl_kind == "scalar":
        dl = np.array([1.7], np.float32)
    else:
        dl = np.random.default_rng(9).uniform(-2, 2, rp.shape).astype(np.float32)
    dld = torch.from_numpy(dl).cuda()
    grad = va.image_loss_backward(pd, gd, dld, cfg, coeffs)
    regrad = va.image_loss_backward(pd, gd, dld, cfg)            # coefficients recomputed
    want = po.image_loss_backward(pred, gt, ocfg, dl, rc)
    np.testing.assert_array_equal(grad.cpu().numpy().view(np.uint32), want.view(np.uint32))
    np.testing.assert_array_equal(regrad.cpu().numpy().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("opts", OPTS)
def test_loss_parity_small(opts):
    pred, gt = _case(37, 53, 4, 1)
    _check(pred, gt, opts, "scalar")
    _check(pred, gt, opts, "partials")


def test_loss_parity_three_channels():
    pred, gt = _case(50, 31, 3, 2)
    _check(pred, gt, dict(), "partials")


def test_loss_parity_rendered_1080p():
    """The loss of a 1920x1080 render of 20k splats against a seeded target."""
    w = scenes.workload("c2", 20_000)
    cam = w.cameras[0].uniforms(w.img_size)
    t, s, o = to_gpu(w.scene)
    out = va.render(cam, w.img_size, t, s, o, pass_=va.RasterPass.BACKWARD)
    pred = out.out_img.cpu().numpy()
    target = scenes.loss_target(w.img_size)
    gt_rgba = np.concatenate([target, np.ones(target.shape[:2] + (1,), np.float32)], -1)
    gt = va.pack_rgba8(torch.from_numpy(gt_rgba)).numpy().view(np.uint32)
    _check(pred, gt, dict(alpha_weight=0.0), "scalar")
    out.state.free()


@pytest.mark.parametrize("cfg", ["c3", "c5"])
def test_l1_cotangent_matches_closed_form(cfg):
    """vs_l1_cotangent (crates/splat-train-loss/src/lib.rs:786-811 sign,
    :1297-1300 weights) at the workload's full image size, with C5's circular
    mask of r = 940 px: bit-equal to sign(pred - gt) / (3 count) on rgb, 0 on
    alpha and on every masked pixel; ties (pred == gt) give 0.  Repeated calls
    (the mask count is cached) give the same result."""
    from tests._util import circle_mask, l1_cotangent_np
    w = scenes.workload(cfg, 1000)
    W, H = w.img_size
    rng = np.random.default_rng(7)
    gt = scenes.loss_target(w.img_size)
    pred = rng.uniform(0, 1, (H, W, 4)).astype(np.float32)
    pred[::7, ::5, :3] = gt[::7, ::5]                                 # exact ties
    mask = circle_mask(w.img_size, w.mask_center, w.mask_radius) if w.mask_radius > 0 else None
    print(f"[case] l1 cotangent {cfg} {W}x{H} mask_radius={w.mask_radius}", flush=True)
    p, g = torch.from_numpy(pred).cuda(), torch.from_numpy(gt).cuda()
    for _ in range(2):
        got = va.l1_cotangent(p, g, w.mask_center, w.mask_radius).cpu().numpy()
        want = l1_cotangent_np(pred, gt, mask)
        np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    assert (got[..., 3] == 0).all() and (got[..., :3][pred[..., :3] == gt] == 0).all()
    if mask is not None:
        assert 0 < mask.mean() < 1 and (got[mask == 0].view(np.uint32) == 0).all()
        assert (got[mask == 1][:, :3] != 0).mean() > 0.9
    # the 12-channel geometry render (surfel training): rgb as above, the other 9 channels 0
    pred12 = np.concatenate([pred, rng.uniform(0, 1, (H, W, 8)).astype(np.float32)], axis=-1)
    got12 = va.l1_cotangent(torch.from_numpy(pred12).cuda(), g, w.mask_center, w.mask_radius).cpu().numpy()
    want12 = np.zeros_like(pred12)
    want12[..., :4] = want
    np.testing.assert_array_equal(got12.view(np.uint32), want12.view(np.uint32))


def test_l1_cotangent_packed_target_matches_unpacked():
    """vs_l1_cotangent_packed reads the reference's u32 RGBA8 target
    (crates/splat-train-loss/src/lib.rs:93,1042-1044: byte x (1/255) in f32):
    bit-equal to vs_l1_cotangent on the float target byte * float32(1/255) and
    to the closed form, with ties at every 7th row, at C5's image size and
    mask, for 4- and 3-channel predictions."""
    from tests._util import circle_mask, l1_cotangent_np
    w = scenes.workload("c5", 1000)
    W, H = w.img_size
    rng = np.random.default_rng(11)
    rgba8 = rng.integers(0, 256, (H, W, 4), dtype=np.uint8)
    gt = rgba8[..., :3].astype(np.float32) * np.float32(1.0 / 255.0)
    pred = rng.uniform(0, 1, (H, W, 4)).astype(np.float32)
    pred[::7, :, :3] = gt[::7]                                         # exact ties
    mask = circle_mask(w.img_size, w.mask_center, w.mask_radius)
    print(f"[case] l1 cotangent packed {W}x{H} mask_radius={w.mask_radius}", flush=True)
    gtp = va.pack_rgba8(torch.from_numpy(rgba8)).cuda()
    assert gtp.dtype == torch.int32 and tuple(gtp.shape) == (H, W)
    want = l1_cotangent_np(pred, gt, mask)
    for c in (4, 3):
        p = torch.from_numpy(np.ascontiguousarray(pred[..., :c])).cuda()
        got = va.l1_cotangent(p, gtp, w.mask_center, w.mask_radius).cpu().numpy()
        ref = va.l1_cotangent(p, torch.from_numpy(gt).cuda(), w.mask_center, w.mask_radius).cpu().numpy()
        np.testing.assert_array_equal(got.view(np.uint32), ref.view(np.uint32))
        np.testing.assert_array_equal(got.view(np.uint32), want[..., :c].view(np.uint32))
    assert (got[::7][..., :3] == 0).all()
    with pytest.raises(ValueError):
        va.l1_cotangent(p, gtp[:, :-1], w.mask_center, w.mask_radius)


@pytest.mark.parametrize("cfg,pass_", [("c3", "BACKWARD"), ("c5", "BACKWARD"), ("c1", "BACKWARD_SMOOTH_CUTOFF")])
def test_forward_fused_l1_cotangent(cfg, pass_):
    """vs_render_forward_l1: the raster pass writes the L1 cotangent of its own
    image (crates/splat-train-loss/src/lib.rs:786-811) bit for bit as
    vs_l1_cotangent_packed computes it from that image, at the workload's full
    size and mask (C5: r = 940), and the image, aux outputs and gradients of
    the render are those of a plain render."""
    w = scenes.workload(cfg, 1000 if cfg == "c1" else 200_000)
    W, H = w.img_size
    rng = np.random.default_rng(5)
    rgba8 = rng.integers(0, 256, (H, W, 4), dtype=np.uint8)
    gtp = va.pack_rgba8(torch.from_numpy(rgba8)).cuda()
    cam = w.cameras[0].uniforms(w.img_size)
    t, s, o = to_gpu(w.scene)
    p = va.RasterPass[pass_]
    print(f"[case] fused l1 {cfg} {W}x{H} {pass_} mask_radius={w.mask_radius}", flush=True)
    fused = va.render(cam, w.img_size, t, s, o, pass_=p, l1_target=gtp, l1_mask_center=w.mask_center,
                      l1_mask_radius=w.mask_radius)
    plain = va.render(cam, w.img_size, t, s, o, pass_=p)
    np.testing.assert_array_equal(fused.out_img.cpu().numpy().view(np.uint32), plain.out_img.cpu().numpy().view(np.uint32))
    for name in ("visible", "max_radius", "opacities", "tile_offsets"):
        np.testing.assert_array_equal(getattr(fused.aux, name).cpu().numpy(), getattr(plain.aux, name).cpu().numpy(),
                                      err_msg=name)
    want = va.l1_cotangent(plain.out_img, gtp, w.mask_center, w.mask_radius)
    got = fused.v_l1
    assert got.shape == (H, W, 4)
    np.testing.assert_array_equal(got.cpu().numpy().view(np.uint32), want.cpu().numpy().view(np.uint32))
    assert (got[..., :3] != 0).float().mean().item() > 0.5
    g1 = va.render_backward(fused, t, s, o, got)
    g2 = va.render_backward(plain, t, s, o, want)
    a, b = g1.v_transforms.cpu().numpy(), g2.v_transforms.cpu().numpy()
    assert (np.abs(a - b) <= 1e-5 + 1e-3 * np.abs(b)).all()
    fused.state.free()
    plain.state.free()


def test_forward_fused_l1_rejects_other_passes():
    w = scenes.workload("c1", 500)
    W, H = w.img_size
    gtp = torch.zeros((H, W), dtype=torch.int32, device="cuda")
    cam = w.cameras[0].uniforms(w.img_size)
    t, s, o = to_gpu(w.scene)
    for p in (va.RasterPass.FORWARD, va.RasterPass.GEOMETRY):
        with pytest.raises(ValueError):
            va.render(cam, w.img_size, t, s, o, pass_=p, l1_target=gtp)
    with pytest.raises(ValueError):
        va.render(cam, w.img_size, t, s, o, pass_=va.RasterPass.BACKWARD, l1_target=gtp[:, :-1])
    with pytest.raises(ValueError):
        va.render(cam, w.img_size, t, s, o, pass_=va.RasterPass.BACKWARD, l1_target=gtp,
                  render_mode=va.SplatRenderMode.SURFEL)


@pytest.mark.parametrize("h,w,cn,opts", [
    (1, 1, 4, dict(mask=True, alpha_weight=0.2)), (5, 64, 3, dict()), (16, 65, 4, dict(alpha_weight=0.3)),
    (17, 63, 3, dict(mask=True)), (33, 59, 4, dict(composite_bg=(0.1, 0.9, 0.4), alpha_weight=0.1)),
    (15, 133, 4, dict(mask=True)), (1040, 2753, 4, dict(mask=True, alpha_weight=0.1)), (2161, 3845, 3, dict()),
])
def test_loss_strips(h, w, cn, opts):
    """The 64-column strips' edges (a column or a row alone, one lane past a
    strip, halo columns cut on either side), with strips of 16 rows (the small
    images) and of several tile rows (the two large ones)."""
    pred, gt = _case(h, w, cn, h + w)
    _check(pred, gt, opts, "partials" if h < 100 else "scalar")
