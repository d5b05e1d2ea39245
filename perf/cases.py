"""The work a program of this library has it do, as measured cases.

A case is one pass through the public entry points of `vauss_amd`: a training
view of a splat cloud (render, loss cotangent, dense gradients) in the sizes of
the five benchmark workloads, a trainer's whole fused step, a surfel view, a
view with the neural appearance, a camera-refinement step, a viewer frame, the
image loss of one frame, and the sort and scan the library exports.  The clouds
have the distributions of `vauss_amd.scenes` (`front` c1 and c2, `orbit` c3,
`heavy` c4, `shell` c5), made on the GPU from a seed.

`exact` restates each computed output in float64 torch, without the library's
code; camera uniforms are inputs like any other.
"""
from __future__ import annotations

import math

import torch

import vauss_amd as va
from vauss_amd.camera import look_at_rotation

DEV = "cuda:0"
TILE = 16

# Camera focal length in units of the image width: c1 256/256, c2 and c3
# 1600/1920, c4 2000/2560, c5 600/1920.
FOCAL = {"small": 1.0, "front": 1600 / 1920, "orbit": 1600 / 1920, "heavy": 2000 / 2560, "shell": 600 / 1920}


def _view(name, scene, n, w, h, sh=3, lagged=True, **more):
    c = {"name": name, "kind": "view", "scene": scene, "n": n, "w": w, "h": h, "sh": sh, "lagged": lagged,
         "model": "pinhole", "mode": "default", "half": False}
    c.update(more)
    return c


def listed():
    return [
        # the smallest benchmark workload, c1: an interactive preview or a unit scene, one waiting (exact-count) render a step
        _view("view_10k_256", "small", 10_000, 256, 256, sh=0, lagged=False),
        # c2: the first thousand steps of a training run, before densification
        _view("view_200k_1080p", "front", 200_000, 1920, 1080),
        # c3: the headline workload, a training view of a densified cloud
        _view("view_1m_1080p", "orbit", 1_000_000, 1920, 1080),
        # c5: training on a fisheye capture, loss inside the lens circle
        _view("view_2m_fisheye", "shell", 2_000_000, 1920, 1920, model="kb4"),
        # c4: a cloud with heavy-tailed scales, as early training and unpruned captures have; every pair is listed (the default)
        _view("view_3m_heavy_1440p", "heavy", 3_000_000, 2560, 1440),
        # one step of the trainer: fused-update render, L1 + SSIM, raster backward, projection VJP + Adam, SH step on f16
        {"name": "step_1m_1080p", "kind": "step", "scene": "orbit", "n": 1_000_000, "w": 1920, "h": 1080, "sh": 3,
         "lagged": True, "model": "pinhole", "mode": "default", "half": True},
        # a 2DGS training view (12 channels, 17 raster gradients), on an image whose sides are no multiple of a tile
        _view("surfel_400k_odd", "orbit", 400_000, 1557, 1037, mode="surfel"),
        # a training view with the compact neural appearance
        {"name": "neural_600k_1080p", "kind": "neural", "scene": "orbit", "n": 600_000, "w": 1920, "h": 1080, "sh": 1,
         "lagged": True, "model": "pinhole", "mode": "default", "half": False, "band": 3},
        # refining the camera of one photo against a trained cloud, anti-aliased (Mip mode with the 3D filter's floor)
        {"name": "pose_300k_odd", "kind": "pose", "scene": "orbit", "n": 300_000, "w": 1237, "h": 823, "sh": 3,
         "lagged": False, "model": "pinhole", "mode": "mip", "half": False},
        # one frame of a viewer: packed RGBA8, Mip mode, f16 coefficients, no backward state
        {"name": "frame_1m_1440p", "kind": "frame", "scene": "orbit", "n": 1_000_000, "w": 2560, "h": 1440, "sh": 3,
         "lagged": False, "model": "pinhole", "mode": "mip", "half": True},
        # the image loss of a training frame with an alpha channel and a mask, at 4K (a trainer that keeps its own optimizer)
        {"name": "loss_4k_rgba", "kind": "loss", "w": 3840, "h": 2160, "channels": 4},
        # the exported sort and scan at the sort crate's large test size
        {"name": "sort_scan_30m", "kind": "sort", "n": 30_000_000, "bits": 32},
    ]


def _odd(rng, lo, hi):
    """An integer spread evenly over the logarithm of [lo, hi], odd more often than not."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, min(hi, v | 1 if rng.random() < 0.7 else v))


def draw(rng):
    kind = rng.choice(["view", "view", "view", "step", "surfel", "neural", "pose", "frame", "loss", "sort"])
    if kind == "sort":
        return {"kind": "sort", "n": _odd(rng, 1000, 30_000_000), "bits": rng.choice([13, 16, 20, 27, 32])}
    if kind == "loss":
        return {"kind": "loss", "w": _odd(rng, 160, 3840), "h": _odd(rng, 120, 2160), "channels": rng.choice([3, 4])}
    c = {"kind": kind, "scene": "orbit", "model": "pinhole", "mode": "default", "half": False, "sh": rng.choice([0, 1, 2, 3]),
         "lagged": rng.random() < 0.5, "w": _odd(rng, 200, 1920), "h": _odd(rng, 150, 1080), "n": _odd(rng, 5000, 1_000_000)}
    if kind == "view":
        c["scene"] = rng.choice(["small", "front", "orbit", "heavy", "shell"])
        c["mode"] = rng.choice(["default", "mip"])
        c["half"] = rng.random() < 0.3
        if c["scene"] == "shell":
            c["model"] = "kb4"
            c["h"] = c["w"]
        if c["scene"] == "heavy":
            c.update(n=_odd(rng, 5000, 3_000_000), w=_odd(rng, 200, 2560), h=_odd(rng, 150, 1440), mode="default")
    elif kind == "step":
        c.update(half=True, lagged=True, n=_odd(rng, 20_000, 1_000_000))
    elif kind == "surfel":
        c.update(kind="view", mode="surfel", n=_odd(rng, 5000, 400_000))
    elif kind == "neural":
        c.update(sh=1, band=rng.choice([0, 1, 2, 3]))
    elif kind == "pose":
        c.update(lagged=False, mode=rng.choice(["default", "mip"]))
    elif kind == "frame":
        c.update(lagged=False, mode=rng.choice(["default", "mip"]), half=rng.random() < 0.5)
    return c


# ---- inputs ---------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 2654435761 % (1 << 62) + 17)
    return g


def _cloud(case, g):
    """(transforms, sh_coeffs, raw_opacities) of the case's scene: vauss_amd.scenes' distributions."""
    n, k, scene = case["n"], (case["sh"] + 1) ** 2, case["scene"]

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=DEV)

    def uniform(*shape):
        return torch.rand(*shape, generator=g, device=DEV)

    ls, raw = normal(n, 3) * 0.7 - 4.5, normal(n) * 1.5
    if scene == "small":
        means = uniform(n, 3) * torch.tensor([2.0, 2.0, 4.0], device=DEV) + torch.tensor([-1.0, -1.0, 2.0], device=DEV)
        ls, raw = normal(n, 3) * 0.5 - 4.0, normal(n)
    elif scene == "front":
        means = normal(n, 3) * 2.0
        means[:, 2] = (means[:, 2] + 7.5).clamp(3.0, 12.0)
    elif scene == "orbit":
        means = normal(n, 3) * 2.0
    elif scene == "heavy":
        means = normal(n, 3) * 1.5
        means[:, 2] = (means[:, 2] + 6.0).clamp(2.0, 10.0)
        ls, raw = normal(n, 3) - 3.0, normal(n) + 1.0
    else:
        means = torch.nn.functional.normalize(normal(n, 3), dim=1) * (uniform(n, 1) * 5.0 + 3.0)
    quats = torch.nn.functional.normalize(normal(n, 4), dim=1)
    sh = normal(n, k, 3) * 0.05
    sh[:, 0] = uniform(n, 3)
    if case["half"]:
        sh = sh.half()
    return torch.cat([means, quats, ls], dim=1).contiguous(), sh, raw


def _camera(case, seed):
    w, h, scene = case["w"], case["h"], case["scene"]
    f = FOCAL[scene] * w
    if scene == "orbit":        # one pose of the radius-6 orbit
        az, el = 2 * math.pi * (seed % 8) / 8 + 0.05 * (seed % 5), math.radians((seed * 7) % 31 - 15)
        pos = [6 * math.cos(el) * math.sin(az), -6 * math.sin(el), -6 * math.cos(el) * math.cos(az)]
        cam = va.Camera.from_focal(f, f, (w, h), position=pos, rotation=look_at_rotation(pos))
    elif case["model"] == "kb4":
        cam = va.Camera.from_focal(f, f, (w, h), model=va.KannalaBrandt4(0.021, -0.017, 0.033, -0.008))
    else:
        cam = va.Camera.from_focal(f, f, (w, h))
    return cam.uniforms((w, h))


def _picture(w, h, g):
    """A smooth RGBA photo with some grain in [0, 1], [h,w,4]; alpha mostly 1."""
    low = torch.rand(1, 4, 12, 16, generator=g, device=DEV)
    img = torch.nn.functional.interpolate(low, size=(h, w), mode="bilinear", align_corners=False)[0].permute(1, 2, 0)
    img = img + 0.04 * torch.randn(h, w, 4, generator=g, device=DEV)
    img[..., 3] = (img[..., 3] * 3).clamp(0, 1)
    return img.clamp(0, 1)


def _packed(img):
    """[h,w,4] in [0, 1] as RGBA8 words, r in the low byte."""
    b = (img * 255.0).round().to(torch.int64)
    p = b[..., 0] | (b[..., 1] << 8) | (b[..., 2] << 16) | (b[..., 3] << 24)
    return torch.where(p >= 1 << 31, p - (1 << 32), p).to(torch.int32).contiguous()


def _mask(case):
    """The fisheye's image circle (940 of 1920 pixels); no mask for other lenses."""
    if case.get("model") != "kb4":
        return (0.0, 0.0), 0.0
    return (case["w"] / 2, case["h"] / 2), case["w"] * 940 / 1920


BETA1, BETA2, EPS, STEP = 0.9, 0.999, 1e-15, 4000
# the means' rate late in its decay, the other rates as 3DGS trains: mean 3, quaternion 4, log-scale 3
LR = [1.6e-6] * 3 + [1e-4] * 4 + [5e-4] * 3
LR_OPAC, LR_SH = 5e-3, 2.5e-4


def _inputs(case, seed):
    g = _gen(seed)
    if case["kind"] == "sort":
        n, bits = case["n"], case["bits"]
        keys = torch.randint(0, 1 << bits, (n,), generator=g, device=DEV, dtype=torch.int64)
        keys = torch.where(keys >= 1 << 31, keys - (1 << 32), keys).to(torch.int32)
        return {"keys": keys, "values": torch.arange(n, dtype=torch.int32, device=DEV),
                "counts": torch.randint(0, 40, (n,), generator=g, device=DEV, dtype=torch.int32)}
    s = {}
    if case["kind"] == "loss":
        target = _picture(case["w"], case["h"], g)
        noise = 0.1 * torch.randn(target.shape, generator=g, device=DEV)
        s["pred"] = (target + noise)[..., :case["channels"]].contiguous()
        s["target"] = _packed(target)
        return s
    s["transforms"], s["sh"], s["raw"] = _cloud(case, g)
    s["cam"] = _camera(case, seed)
    s["size"] = (case["w"], case["h"])
    s["mask_center"], s["mask_radius"] = _mask(case)
    if case["kind"] != "frame":
        s["target"] = _packed(_picture(case["w"], case["h"], g))
    n = case["n"]
    if case["mode"] == "mip":
        s["floor"] = torch.rand(n, generator=g, device=DEV) * 0.01 + 0.001
    if case["kind"] == "neural":
        s["sh"] = torch.rand(n, 4, 3, generator=g, device=DEV) * 3.0 - 1.5
        s["decoder"] = torch.randn(816, generator=g, device=DEV) * 0.35
    if case["kind"] == "step":
        def moments(*shape):        # a warm optimizer: |m| of the order of sqrt(v), over a few decades of sizes
            v = torch.exp(torch.randn(*shape, generator=g, device=DEV) * 2.0 - 16.0)
            return torch.randn(*shape, generator=g, device=DEV) * 0.3 * v, v * v
        s["geo"], s["geo_opac"] = moments(n, 10), moments(n)
        k3 = s["sh"].shape[1] * 3
        s["sh_m"] = torch.randn(n, k3, generator=g, device=DEV) * 1e-7
        s["sh_v"] = torch.exp(torch.randn(n, generator=g, device=DEV) - 32.0)
    return s


_MODES = {"default": va.SplatRenderMode.DEFAULT, "mip": va.SplatRenderMode.MIP, "surfel": va.SplatRenderMode.SURFEL}


def _pass(case):
    return {"frame": va.RasterPass.FORWARD, "step": va.RasterPass.BACKWARD_FUSED_UPDATE}.get(case["kind"],
                                                                                             va.RasterPass.BACKWARD)


def _render(s, **more):
    return va.render(s["cam"], s["size"], s["transforms"], s["sh"], s["raw"], pass_=s["pass"], render_mode=s["mode"],
                     min_scale=s.get("floor"), decoder=s.get("decoder"), neural_degree=s.get("band", 0), **more)


def prepare(case, seed):
    s = _inputs(case, seed)
    s["kind"] = case["kind"]
    if case["kind"] == "sort":
        s["bits"] = case["bits"]
        return s
    if case["kind"] == "loss":
        alpha = case["channels"] == 4
        s["cfg"] = va.ImageLossConfig(0.8, -0.2, mask=alpha, alpha_weight=0.1 if alpha else 0.0)
        s["one"] = torch.ones(1, device=DEV)
        return s
    s["pass"], s["mode"], s["band"] = _pass(case), _MODES[case["mode"]], case.get("band", 0)
    if case["kind"] == "step":
        s["cfg"], s["one"] = va.ImageLossConfig.l1_dssim(0.2), torch.ones(1, device=DEV)
        s["w_t"], s["w_o"] = va.geo_encode(*s.pop("geo"), EPS), va.geo_encode(*s.pop("geo_opac"), EPS)
        s["lr"] = torch.tensor(LR, device=DEV)
        s["sh_state"] = va.ShStepState(va.Block8Moment.encode(s.pop("sh_m")), s.pop("sh_v"), STEP - 1)
        s["lr_sh"] = torch.ones(s["sh"].shape[1] * 3, device=DEV)
        s["lr_sh"][3:] = 1 / 20
        s["adam"] = va.FusedAdam.at_step(STEP, lr_opac=LR_OPAC, beta1=BETA1, beta2=BETA2, epsilon=EPS)
    # a trainer turns lagged counts on once; an exact render first, as its evaluation renders are, fits the capacity
    ctx = va.Context.get(torch.device(DEV))
    ctx.set_lagged_counts(False)
    if case["lagged"]:
        out = _render(s)
        if out.state is not None:
            out.state.free()
        ctx.set_lagged_counts(True)
    return s


# ---- one pass ----------------------------------------------------------------------

def run(s):
    if s["kind"] == "sort":
        keys, order = va.radix_argsort(s["keys"], s["values"], s["bits"])
        return {"keys": keys, "order": order, "offsets": va.prefix_sum(s["counts"])}
    if s["kind"] == "loss":
        partials, coeffs, total = va.image_loss_forward_train(s["pred"], s["target"], s["cfg"])
        v = va.image_loss_backward(s["pred"], s["target"], s["one"], s["cfg"], coeffs)
        return {"partials": partials, "coeffs": coeffs, "total": total, "v_pred": v}
    if s["kind"] == "frame":
        out = _render(s)
        return {"image": out.out_img, "max_radius": out.aux.max_radius, "opacities": out.aux.opacities}
    t, sh, raw = s["transforms"], s["sh"], s["raw"]
    if s["kind"] == "step":
        out = _render(s)
        _, coeffs, total = va.image_loss_forward_train(out.out_img, s["target"], s["cfg"])
        v = va.image_loss_backward(out.out_img, s["target"], s["one"], s["cfg"], coeffs)
        g = va.render_backward(out, t, sh, raw, v)
        up = va.project_update(out, t, sh, raw, g.v_combined, s["w_t"], s["lr"], s["w_o"], s["adam"])
        out.state.free()
        va.sh_step(sh, up.color_dir, up.compact_from_global, up.coeffs_grad_sq, s["sh_state"], LR_SH, s["lr_sh"],
                   BETA1, BETA2, EPS)
        return {"image": out.out_img, "total": total, "v_image": v, "v_combined": g.v_combined,
                "transforms": t, "raw": raw, "w_t": s["w_t"], "w_o": s["w_o"], "color_dir": up.color_dir,
                "refine": up.v_refine_weight, "sh": sh, "variance": s["sh_state"].variance,
                "codes": s["sh_state"].moment.codes, "scales": s["sh_state"].moment.scales}
    if s["mode"] is va.SplatRenderMode.SURFEL:
        out = _render(s)
        v = va.l1_cotangent(out.out_img, s["target"], s["mask_center"], s["mask_radius"])
    else:
        out = _render(s, l1_target=s["target"], l1_mask_center=s["mask_center"], l1_mask_radius=s["mask_radius"])
        v = out.v_l1
    g = va.render_backward(out, t, sh, raw, v, min_scale=s.get("floor"), decoder=s.get("decoder"))
    r = {"image": out.out_img, "v_image": v, "visible": out.aux.visible, "max_radius": out.aux.max_radius,
         "opacities": out.aux.opacities, "tile_offsets": out.aux.tile_offsets, "v_transforms": g.v_transforms,
         "v_coeffs": g.v_coeffs, "v_raw": g.v_raw_opac, "refine": g.v_refine_weight, "v_combined": g.v_combined}
    if s["kind"] == "neural":
        r["v_decoder"], r["v_coeffs_sq"] = g.v_decoder, g.v_coeffs_sq
    if s["kind"] == "pose":
        r["v_pose"] = va.pose_backward(out, t, sh, raw, g.v_combined, min_scale=s.get("floor"))
    out.state.free()
    return r


def work(case):
    """Inputs read once and outputs written once; operations of about 80 blended splats a pixel, 25 each forward and 75 backward."""
    if case["kind"] == "sort":
        return {"bytes": case["n"] * 24, "flops": 0}
    px = case["w"] * case["h"]
    if case["kind"] == "loss":      # 22 taps of 5 moments forward and 3 coefficients backward, three channels
        return {"bytes": px * (2 * (4 * case["channels"] + 4) + 2 * 36 + 4 * case["channels"]), "flops": px * 3 * 2 * 22 * 8}
    n, k3 = case["n"], 3 * (case["sh"] + 1) ** 2
    shb = 2 if case["half"] else 4
    read = n * (44 + 0.6 * shb * k3)
    if case["kind"] == "frame":
        return {"bytes": read + 4 * px + 8 * n, "flops": px * 80 * 25}
    if case["kind"] == "step":      # + image, its gradient, both again; parameters, two moments, coefficients and codes back
        return {"bytes": read + n * (40 + 88 + 44 + 24 + 8 + 4 + k3 * 4) + px * 40 + px * 88, "flops": px * 80 * 100}
    ch, gr = (12, 17) if case["mode"] == "surfel" else (4, 10)
    return {"bytes": read + n * (48 + 4 * k3 + 4 * gr + 12) + px * (8 * ch + 4), "flops": px * 80 * 100 * (3 if ch == 12 else 1)}


def tolerance(case):
    if case["kind"] in ("sort", "frame"):
        return "exact"
    if case["kind"] == "loss":      # window sums in another order, amplified by the variances' cancellation
        return {"rel": 1e-3, "max": 0.1}
    # gradients are sums of f32 atomics in a run's own order; a pixel whose cotangent or cut flips moves one splat's row
    return {"rel": 2e-3, "max": 0.3, "differ": 0.005}


# ---- the same in float64 ---------------------------------------------------------------

SH_C0 = 0.28209479177387814


def _basis(v, degree):
    """Real spherical harmonics of unit directions [n,3], [n,(degree+1)^2], in the coefficients' order and signs."""
    x, y, z = v.unbind(1)
    y_ = [torch.full_like(x, SH_C0)]
    if degree >= 1:
        c = math.sqrt(3 / (4 * math.pi))
        y_ += [-c * y, c * z, -c * x]
    if degree >= 2:
        c = math.sqrt(15 / (4 * math.pi))
        y_ += [c * x * y, -c * y * z, math.sqrt(5 / (16 * math.pi)) * (3 * z * z - 1), -c * x * z, 0.5 * c * (x * x - y * y)]
    if degree >= 3:
        a, b = math.sqrt(35 / (32 * math.pi)), math.sqrt(105 / (4 * math.pi))
        c, d = math.sqrt(21 / (32 * math.pi)), math.sqrt(7 / (16 * math.pi))
        y_ += [-a * y * (3 * x * x - y * y), b * x * y * z, -c * y * (5 * z * z - 1), d * z * (5 * z * z - 3),
               -c * x * (5 * z * z - 1), 0.5 * b * z * (x * x - y * y), -a * x * (x * x - 3 * y * y)]
    return torch.stack(y_, dim=1)


def _ge0(x):
    """max(x, 0) whose slope at 0 is 1, the colours' gate."""
    return torch.where(x >= 0, x, torch.zeros_like(x))


def _rotations(q):
    w, x, y, z = torch.nn.functional.normalize(q, dim=1).unbind(1)
    return torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                        2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                        2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], dim=1).view(-1, 3, 3)


class _Proj:
    """Differentiable projection of the kept splats: `keep` ids, raster rows, binning ellipse, depth."""


def _project(case, s, t, sh, raw, decoder, pose=None):
    cam, (w, h) = s["cam"], s["size"]
    V = torch.tensor(list(cam.viewmat), dtype=torch.float64, device=DEV).view(4, 3)
    R, tr = V[:3].t(), V[3]
    eye = torch.tensor(list(cam.cam_pos), dtype=torch.float64, device=DEV)
    surfel, mip = case["mode"] == "surfel", case["mode"] == "mip"
    with torch.no_grad():
        mc = t[:, :3] @ R.t() + tr
        if cam.model == 0:
            front = mc[:, 2] >= 0.01
        else:
            front = torch.atan2(mc[:, :2].norm(dim=1), mc[:, 2]) <= cam.half_max_render_fov
    p = _Proj()
    keep = front.nonzero()[:, 0]
    for last in (False, True):      # the second time over the splats that pass every cull
        means, q, ls = t[keep, :3], t[keep, 3:7], t[keep, 7:]
        xc = means @ R.t() + tr
        if pose is not None:
            xc = xc + xc @ pose[:9].view(3, 3).t() + pose[9:]
        scale, opac = ls.exp(), torch.sigmoid(raw[keep])
        if "floor" in s:
            floored = (scale * scale + s["floor"][keep].double()[:, None] ** 2).sqrt()
            opac = (opac * (scale / floored).prod(dim=1)).clamp(1e-6, 1 - 1e-6)
            scale = floored
        if not last:
            p.opacities = torch.zeros(case["n"], dtype=torch.float64, device=DEV).index_put((keep,), opac.detach())
        rot = R @ _rotations(q)
        if pose is not None:
            rot = rot + pose[:9].view(3, 3) @ rot
        x, y, z = xc.unbind(1)
        if surfel:
            K = torch.tensor([[cam.fx, 0, cam.cx], [0, cam.fy, cam.cy], [0, 0, 1]], dtype=torch.float64, device=DEV)
            M = torch.stack([rot[:, :, 0] * scale[:, :1], rot[:, :, 1] * scale[:, 1:2], xc], dim=2)
            M = K @ M
            power = (opac * 255).log()
            k2 = torch.stack([2 * power, 2 * power, -torch.ones_like(power)], dim=1)
            D = (M * k2[:, None]) @ M.transpose(1, 2)
            nrm = -D[:, 2, 2]
            x0, y0 = -D[:, 0, 2] / nrm, -D[:, 1, 2] / nrm
            s00, s01, s11 = D[:, 0, 0] / nrm + x0 * x0, D[:, 0, 1] / nrm + x0 * y0, D[:, 1, 1] / nrm + y0 * y0
            tt = (0.5 * (s00 + s11)).clamp_min(1e-12).div(power.clamp_min(1e-12)).sqrt().clamp(1e-3, 1e3)
            ga, gb = 1 + 1 / tt, (1 + tt) * power
            ex, ey = (ga * s00 + gb).clamp_min(0).sqrt(), (ga * s11 + gb).clamp_min(0).sqrt()
            ok = (nrm > 1e-12) & (power >= 0) & ((ga * s00 + gb) * (ga * s11 + gb) - (ga * s01) ** 2 > 0)
            cx, cy = x0, y0
            n = rot[:, :, 2]
            n = n * torch.where((n * xc).sum(dim=1) > 0, -1.0, 1.0)[:, None]
            geo = torch.cat([M.reshape(-1, 9), n], dim=1)
        else:
            if cam.model == 0:
                cx, cy = cam.fx * x / z + cam.cx, cam.fy * y / z + cam.cy
                o = torch.zeros_like(z)
                jx, jy = (x / z).clamp(cam.lim_neg_x, cam.lim_pos_x), (y / z).clamp(cam.lim_neg_y, cam.lim_pos_y)
                J = torch.stack([cam.fx / z, o, -cam.fx / z * jx, o, cam.fy / z, -cam.fy / z * jy], dim=1).view(-1, 2, 3)
            else:
                k1, k2, k3, k4 = list(cam.kb4)
                r, rho2 = (x * x + y * y).sqrt(), x * x + y * y + z * z
                th = torch.atan2(r, z)
                a = th * th
                d = th * (1 + a * (k1 + a * (k2 + a * (k3 + a * k4))))
                dd = 1 + a * (3 * k1 + a * (5 * k2 + a * (7 * k3 + a * 9 * k4)))
                f = d / r
                fr, fz = (dd * z / rho2 - f) / r, dd * (-r / rho2) / r
                cx, cy = cam.fx * f * x + cam.cx, cam.fy * f * y + cam.cy
                J = torch.stack([cam.fx * (f + x * x * fr / r), cam.fx * x * y * fr / r, cam.fx * x * fz,
                                 cam.fy * x * y * fr / r, cam.fy * (f + y * y * fr / r), cam.fy * y * fz], dim=1).view(-1, 2, 3)
            A = J @ (rot * scale[:, None])
            c = A @ A.transpose(1, 2)
            blur = 0.1 if mip else 0.3
            a, b, d = c[:, 0, 0] + blur, c[:, 0, 1], c[:, 1, 1] + blur
            det = a * d - b * b
            if mip:     # the compensation is held fixed in the gradient
                opac = opac * ((c[:, 0, 0] * c[:, 1, 1] - b * b).clamp_min(0) / det).sqrt().detach()
            power = (opac * 255).log()
            ex, ey = (2 * power.clamp_min(0) * a).sqrt(), (2 * power.clamp_min(0) * d).sqrt()
            ok = power >= 0
            geo = torch.stack([cx, cy, d / det, -b / det, a / det], dim=1)
        ok = ok & (cx + ex > 0) & (cx - ex < w) & (cy + ey > 0) & (cy - ey < h)
        if not last:
            keep = keep[ok.nonzero()[:, 0]]
    at = eye
    if pose is not None:        # only the camera centre moves the view direction: by -M^-1 b
        at = eye - torch.linalg.solve(R, pose[9:])
    direction = torch.nn.functional.normalize(means - at, dim=1)
    if decoder is not None:
        row = sh[keep].view(-1, 12)
        f = row[:, 3:11]
        band = case["band"]
        basis = _basis(direction, band)
        x_in = torch.cat([torch.stack([f.sin(), f.cos()], dim=2).view(-1, 16), basis], dim=1)
        W1 = decoder[:512].view(16, 32)[:, :16 + basis.shape[1]]
        h1 = torch.relu(x_in @ W1.t())
        h2 = torch.relu(h1 @ decoder[512:768].view(16, 16).t())
        rgb = torch.relu(row[:, :3] * SH_C0 + torch.tanh(h2 @ decoder[768:].view(3, 16).t()) + 0.5)
    else:
        rgb = (_basis(direction, case["sh"])[:, :, None] * sh[keep]).sum(dim=1) + 0.5
    p.keep, p.rows, p.direction = keep, torch.cat([geo, rgb, opac[:, None]], dim=1), direction
    p.depth, p.box = z.detach(), torch.stack([cx - ex, cx + ex, cy - ey, cy + ey], dim=1).detach()
    p.max_radius = torch.zeros(case["n"], dtype=torch.float64, device=DEV)
    p.max_radius[keep] = torch.maximum(ex / w, ey / h).detach()
    return p


MOST_PAIRS = 24_000_000


def _lists(p, w, h):
    """Depth-ordered splats of each tile as (offsets [T+1], splats); None when there are too many."""
    tw, th = (w + TILE - 1) // TILE, (h + TILE - 1) // TILE
    b = (p.box / TILE).floor().to(torch.int64)
    x0, x1 = b[:, 0].clamp(0, tw - 1), b[:, 1].clamp(0, tw - 1)
    y0, y1 = b[:, 2].clamp(0, th - 1), b[:, 3].clamp(0, th - 1)
    cols, count = x1 - x0 + 1, (x1 - x0 + 1) * (y1 - y0 + 1)
    if int(count.sum()) > MOST_PAIRS:
        return None
    # the depth key is the raw bits of z: splats behind a wide lens's plane come last, nearest the plane first
    order = torch.argsort(torch.where(p.depth < 0, 1e30 * (1 - p.depth), p.depth), stable=True)
    splat = torch.repeat_interleave(order, count[order])
    first = torch.cumsum(count[order], 0) - count[order]
    i = torch.arange(splat.numel(), device=DEV) - torch.repeat_interleave(first, count[order])
    tile = (y0[splat] + i // cols[splat]) * tw + x0[splat] + i % cols[splat]
    tile, by = torch.sort(tile, stable=True)
    offsets = torch.searchsorted(tile, torch.arange(tw * th + 1, device=DEV))
    return offsets, splat[by], tw


def _chunks(offsets, values=3_000_000):
    """Groups of tiles whose padded lists hold at most `values` (splat, pixel) pairs: (tiles, longest list)."""
    length = (offsets[1:] - offsets[:-1])
    length, tiles = torch.sort(length, descending=True)
    length = length.tolist()
    i = 0
    while i < len(length):
        k = max(1, min(len(length) - i, values // (256 * max(1, length[i]))))
        yield tiles[i:i + k], length[i]
        i += k


def _composite(case, rows, px, py, bg=0.0):
    """Channels [t,256,C] of padded lists: rows [t,L,k] (opacity 0 pads), pixel centres [t,1,256]."""
    surfel = case["mode"] == "surfel"
    if surfel:
        m = rows[..., :9, None].unbind(2)
        ux, uy, uz = m[0] - px * m[6], m[1] - px * m[7], m[2] - px * m[8]
        vx, vy, vz = m[3] - py * m[6], m[4] - py * m[7], m[5] - py * m[8]
        qx, qy, qz = uy * vz - uz * vy, uz * vx - ux * vz, ux * vy - uy * vx
        miss = qz == 0
        qz = torch.where(miss, torch.ones_like(qz), qz)
        su, sv = qx / qz, qy / qz
        z = m[6] * su + m[7] * sv + m[8]
        dx, dy = px - m[2] / m[8], py - m[5] / m[8]
        sigma = 0.5 * torch.minimum(su * su + sv * sv, 2 * (dx * dx + dy * dy))
        good = ~miss & (z.detach() >= 0.01)
    else:
        x, y, a, b, c = rows[..., :5, None].unbind(2)
        dx, dy = px - x, py - y
        sigma = 0.5 * (a * dx * dx + c * dy * dy) + b * dx * dy
        good = True
    rgb, opac = _ge0(rows[..., -4:-1]), rows[..., -1:]
    alpha = (opac * torch.exp(-sigma)).clamp(max=0.999)
    alpha = torch.where(good & (alpha >= 1 / 255) & (sigma >= 0), alpha, torch.zeros_like(alpha))
    loss = torch.log1p(-alpha)
    after = torch.cumsum(loss, dim=1)
    live = after.detach() > math.log(1e-4)
    before = (after - loss).exp()
    vis = torch.where(live, alpha * before, torch.zeros_like(alpha))
    T = torch.where(live, loss, torch.zeros_like(loss)).sum(dim=1).exp()
    out = [torch.einsum("tlp,tlc->tpc", vis, rgb) + bg * T[..., None], (1 - T)[..., None]]
    if surfel:
        def total(v):
            return (vis * v).sum(dim=1)[..., None]
        z = torch.where(live & (alpha > 0), z, torch.ones_like(z))
        dist = 100.0 / (100.0 - 0.2) * (1 - 0.2 / z.clamp_min(0.2))
        blended = live & (alpha > 0) & (before > 0.5)       # the last of these is the median
        place = torch.arange(1, blended.shape[1] + 1, device=DEV)[None, :, None]
        at = (blended * place).max(dim=1).values
        median = torch.where(at > 0, z.gather(1, (at - 1).clamp_min(0)[:, None])[:, 0], torch.zeros_like(T))
        ident = torch.where(at > 0, torch.zeros_like(T), torch.full_like(T, float("nan")))
        out += [total(z), median[..., None], torch.einsum("tlp,tlc->tpc", vis, rows[..., 9:12]), total(dist), total(dist * dist),
                ident[..., None]]
    return torch.cat(out, dim=2)


def _padded(p, lists, tiles, longest):
    offsets, splats, tw = lists
    lo, n = offsets[tiles], offsets[tiles + 1] - offsets[tiles]
    i = torch.arange(longest, device=DEV)[None]
    pad = i >= n[:, None]
    ids = splats[(lo[:, None] + i).clamp_max(splats.numel() - 1)]
    j = torch.arange(256, device=DEV)
    px = (tiles % tw * TILE)[:, None] + j % TILE
    py = (tiles // tw * TILE)[:, None] + j // TILE
    return ids, pad, px, py


def _image64(case, s, p, lists):
    w, h = s["size"]
    img = torch.zeros(h, w, 12 if case["mode"] == "surfel" else 4, dtype=torch.float64, device=DEV)
    if img.shape[2] == 12:
        img[..., 11] = float("nan")
    rows = p.rows.detach()
    with torch.no_grad():
        for tiles, longest in _chunks(lists[0]):
            if not longest:
                continue
            ids, pad, px, py = _padded(p, lists, tiles, longest)
            r = rows[ids]
            r[..., -1] = torch.where(pad, torch.zeros_like(r[..., -1]), r[..., -1])
            c = _composite(case, r, px[:, None] + 0.5, py[:, None] + 0.5)
            ok = (px < w) & (py < h)
            img[py[ok], px[ok]] = c[ok]
    return img


def _raster_grad(case, s, p, lists, v):
    """Gradients of the kept splats' rows [K,k] and their refine weights [K]."""
    w, h = s["size"]
    rows = p.rows.detach()
    grad = torch.zeros_like(rows)
    refine = torch.zeros(rows.shape[0], dtype=torch.float64, device=DEV)
    v = torch.nan_to_num(v)
    for tiles, longest in _chunks(lists[0]):
        if not longest:
            continue
        ids, pad, px, py = _padded(p, lists, tiles, longest)
        r = rows[ids]
        r[..., -1] = torch.where(pad, torch.zeros_like(r[..., -1]), r[..., -1])
        r.requires_grad_(True)
        # a shift of each (splat, pixel) pair's pixel, for the screen-space gradient before it is summed
        sx = torch.zeros(r.shape[0], longest, 256, dtype=torch.float64, device=DEV, requires_grad=True)
        sy = torch.zeros_like(sx, requires_grad=True)
        c = _composite(case, r, px[:, None] + 0.5 - sx, py[:, None] + 0.5 - sy)
        ok = (px < w) & (py < h)
        cot = torch.where(ok[..., None], v[py.clamp_max(h - 1), px.clamp_max(w - 1)], torch.zeros_like(c))
        c = torch.where(torch.isnan(c), torch.zeros_like(c), c)
        gr, gx, gy = torch.autograd.grad((c * cot).sum(), (r, sx, sy))
        final = c[..., 3].detach().clamp_min(1e-5)
        norm = ((gx * w) ** 2 + (gy * h) ** 2).sqrt() / final[:, None]
        gr = torch.where(pad[..., None], torch.zeros_like(gr), gr)
        grad.index_add_(0, ids.reshape(-1), gr.reshape(-1, gr.shape[-1]))
        refine.index_add_(0, ids.reshape(-1), torch.where(pad[..., None], torch.zeros_like(norm), norm).sum(dim=2).reshape(-1))
    return grad, refine


def _unpacked(target):
    t = target.to(torch.int64)
    return torch.stack([(t >> s) & 255 for s in (0, 8, 16, 24)], dim=2).double() / 255


def _l1(case, s, img):
    h, w = img.shape[:2]
    v = torch.zeros_like(img)
    d = (img[..., :3] - _unpacked(s["target"])[..., :3]).sign()
    if s["mask_radius"] > 0:
        y, x = torch.meshgrid(torch.arange(h, device=DEV) + 0.5, torch.arange(w, device=DEV) + 0.5, indexing="ij")
        inside = (x - s["mask_center"][0]) ** 2 + (y - s["mask_center"][1]) ** 2 <= s["mask_radius"] ** 2
        v[..., :3] = d * inside[..., None] / (3 * int(inside.sum()))
    else:
        v[..., :3] = d / (3 * h * w)
    return v


def _blur(x):
    """11-tap Gaussian window (sigma 1.5) over [c,h,w], zero outside."""
    taps = torch.exp(-((torch.arange(11, dtype=torch.float64, device=DEV) - 5) ** 2) / 4.5)
    taps = (taps / taps.sum()).tolist()
    for dim in (2, 1):
        n = x.shape[dim]
        pad = torch.nn.functional.pad(x, (5, 5) if dim == 2 else (0, 0, 5, 5))
        x = sum(k * pad.narrow(dim, i, n) for i, k in enumerate(taps))
    return x


def _loss(pred, target, l1_weight, ssim_weight, alpha_weight, mask):
    """(partials, coefficients, total, gradient of the total) of the L1 + SSIM loss."""
    h, w, cn = pred.shape
    gt = _unpacked(target).permute(2, 0, 1)
    p = pred.double().permute(2, 0, 1).detach().requires_grad_(True)
    x, y = p[:3], gt[:3]
    mu1, mu2 = _blur(x), _blur(y)
    m11 = _blur(x * x)
    m12 = _blur(x * y)
    s2 = (_blur(y * y) - mu2 * mu2).clamp_min(0)
    s1 = (m11 - mu1 * mu1).clamp_min(0)
    s12 = m12 - mu1 * mu2
    c1, c2 = 1e-4, 9e-4
    a, b, ct, dt = mu1 * mu1 + mu2 * mu2 + c1, s1 + s2 + c2, 2 * mu1 * mu2 + c1, 2 * s12 + c2
    per = l1_weight * (x - y).abs() + ssim_weight * (ct * dt / (a * b)).clamp(-1, 1)
    per = per * (1 / (3.0 * h * w)) * (gt[3] if mask else 1.0)
    if alpha_weight > 0:
        al = (p[3] - gt[3]).abs() * (gt[3] if mask else 1.0) * alpha_weight / (h * w)
        per = torch.cat([per, al[None]])
    total = per.sum()
    grad, = torch.autograd.grad(total, p)
    with torch.no_grad():
        cd = ct * dt / (a * b)
        co = torch.stack([2 / (a * b) * (mu2 * (dt - ct) - mu1 * cd * (b - a)), -cd / b, 2 * ct / (a * b)], dim=1)
        co = torch.where((cd.abs() > 1)[:, None], torch.zeros_like(co), co)
        th, tw = -(-h // TILE), -(-w // TILE)
        tiles = torch.nn.functional.pad(per, (0, tw * TILE - w, 0, th * TILE - h)).view(-1, th, TILE, tw, TILE).sum(dim=(2, 4))
    return tiles.reshape(tiles.shape[0], -1), co, total.detach().view(1), grad.permute(1, 2, 0).contiguous()


def _geo_decode(words):
    """(u, growth) of packed moments: sqrt(v) = eps (growth - 1), m = u eps growth."""
    wd = words.to(torch.int64) & 0xFFFFFFFF
    u = (wd & 0x7FFF).double() * (8 / 32767)
    return torch.where((wd & 0x8000) != 0, -u, u), torch.exp((wd >> 16).double() * (64 / 65535))


def _adam64(param, words, g, lr):
    u, growth = _geo_decode(words)
    m = u * EPS * growth * BETA1 + g * (1 - BETA1)
    v = (EPS * (growth - 1)) ** 2 * BETA2 + g * g * (1 - BETA2)
    return param - lr * (m / (1 - BETA1 ** STEP)) / ((v / (1 - BETA2 ** STEP)).sqrt() + EPS)


def _scatter(n, keep, rows):
    out = torch.zeros((n,) + rows.shape[1:], dtype=torch.float64, device=DEV)
    out[keep] = rows
    return out


def exact(case, seed):
    if case["kind"] == "sort":          # whole numbers
        return None
    if case["kind"] == "loss":
        s, alpha = _inputs(case, seed), case["channels"] == 4
        partials, co, total, v = _loss(s["pred"], s["target"], 0.8, -0.2, 0.1 if alpha else 0.0, alpha)
        return {"partials": partials, "coeffs": co, "total": total, "v_pred": v}
    s = _inputs(case, seed)
    n = case["n"]
    t, sh, raw = (s[k].double().requires_grad_(True) for k in ("transforms", "sh", "raw"))
    decoder = s["decoder"].double().requires_grad_(True) if "decoder" in s else None
    pose = torch.zeros(12, dtype=torch.float64, device=DEV, requires_grad=True) if case["kind"] == "pose" else None
    p = _project(case, s, t, sh, raw, decoder, pose)
    if case["kind"] == "frame":         # the packed image is whole numbers
        return {"image": None, "max_radius": p.max_radius, "opacities": p.opacities}
    lists = _lists(p, *s["size"])
    if lists is None:                   # over 20 seconds
        return None
    img = _image64(case, s, p, lists)
    if case["kind"] == "step":
        _, _, total, v = _loss(img, s["target"], 0.8, -0.2, 0.0, False)
    else:
        v = _l1(case, s, img)
    rows, refine = _raster_grad(case, s, p, lists, v)
    leaves = [x for x in (t, sh, raw, decoder, pose) if x is not None]
    grads = torch.autograd.grad((p.rows * rows).sum(), leaves)
    combined = _scatter(n, p.keep, torch.cat([rows, refine[:, None]], dim=1))
    # a nearly edge-on surfel meets a ray far away, at a depth without a correct digit in 32 bits: its 12 channels have no such value
    r = {"image": None if case["mode"] == "surfel" else img, "v_image": v, "max_radius": p.max_radius, "opacities": p.opacities, "v_transforms": grads[0],
         "v_coeffs": grads[1], "v_raw": grads[2], "refine": _scatter(n, p.keep, refine), "v_combined": combined}
    if case["kind"] == "step":
        color = torch.cat([combined[:, 5:8], _scatter(n, p.keep, p.direction.detach())], dim=1)
        color = torch.where((combined != 0).any(dim=1)[:, None], color, torch.zeros_like(color))
        gsq = (color[:, :3] * SH_C0).square().mean(dim=1)
        seen = _scatter(n, p.keep, torch.ones(p.keep.numel(), dtype=torch.float64, device=DEV))
        var = s["sh_v"].double()
        w_t, w_o = va.geo_encode(*s["geo"], EPS), va.geo_encode(*s["geo_opac"], EPS)    # inputs: the packed moments in hand
        lr = torch.tensor(LR, dtype=torch.float64, device=DEV)
        return {"image": img, "total": total, "v_image": v, "v_combined": combined,
                "transforms": _adam64(t.detach(), w_t, grads[0], lr), "raw": _adam64(raw.detach(), w_o, grads[2], LR_OPAC),
                "color_dir": torch.cat([torch.zeros(1, 6, dtype=torch.float64, device=DEV), color]),
                "refine": _scatter(n, p.keep, refine), "variance": torch.where(seen > 0, var * BETA2 + gsq * (1 - BETA2), var)}
    if case["kind"] == "neural":
        r["v_decoder"], r["v_coeffs_sq"] = grads[3], grads[1].reshape(n, 12).square().mean(dim=1)
    if case["kind"] == "pose":
        r["v_pose"] = grads[-1]
    return r
