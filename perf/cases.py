"""The workloads this framework's speed is judged on, with their inputs, outputs and tolerances.

Every case calls the public entry points as a user's program does: whole frames (``frame.render_frame``,
``frame.render_rig``, ``ut_gs_render``), forward only and as a training step with the gradient of every
leaf, and the layers a program may call by itself (the compositor, the colours, the tile binning). Scenes
follow the distributions of ``xsimgs_amd.synthetic``, drawn on the GPU.

``exact`` restates in float64 torch the pinhole projection, the tile lists and the compositing (and its
gradients) with the thresholds the renderer defines: alpha at least 1/255 and at most 0.999 (0.99 in the
backward), a pixel ending before its transmittance would reach 1e-4.
"""
import math

import torch

DEV = "cuda"


def listed():
    return [
        # a viewer's thumbnail: ten thousand Gaussians, one small image; launches and host time count
        dict(name="view_256", kind="frame", scene="box", n=10_000, width=256, height=256, degree=0, train=False),
        # the viewer's full-size image of a large scene, most of which is out of view
        dict(name="view_1080p", kind="frame", scene="wide", n=1_000_000, width=1920, height=1080, degree=3,
             train=False),
        # one step of training on that scene: the headline frame
        dict(name="train_1080p", kind="frame", scene="wide", n=1_000_000, width=1920, height=1080, degree=3,
             train=True),
        # a training step on a smaller scene and an odd image size, every Gaussian in view
        dict(name="train_odd", kind="frame", scene="frustum", n=150_001, width=1237, height=701, degree=2,
             train=True),
        # a spinning lidar's range image: intensity and ray-drop channels, phase modelling, 32x8 tiles
        dict(name="train_lidar", kind="lidar", n=3_000_000, width=2048, height=128, train=True),
        # a driving rig: six cameras at one origin over one scene, batched
        dict(name="train_rig", kind="rig", n=4_000_000, width=1600, height=900, cameras=6, train=True),
        # a rolling-shutter camera on a moving vehicle, moving Gaussians: per-pixel origins and times
        dict(name="train_rolling", kind="render", lens="pinhole", n=400_000, width=1280, height=800, shutter=True,
             motion=True, train=True),
        # a fisheye lens, odd image size, forward only
        dict(name="view_fisheye", kind="render", lens="fisheye", n=500_003, width=1501, height=999, shutter=False,
             motion=False, train=False),
        # the compositor by itself: a training step that also refines the camera's pose (ray gradients)
        dict(name="raster_pose", kind="raster", n=60_000, width=800, height=600, channels=3, tile_x=16, tile_y=16,
             motion=False, ray_grads=True),
        # the compositor with a feature vector per Gaussian instead of a colour
        dict(name="raster_features", kind="raster", n=50_000, width=640, height=480, channels=32, tile_x=16,
             tile_y=16, motion=False, ray_grads=False),
        # view-dependent colours of a large model in the other layout, forward and backward
        dict(name="colours_3kn", kind="colours", n=1_500_000, degree=3, layout_3kn=True, dc=False, masked=False),
        # the tile lists by themselves, with the 64-bit keys
        dict(name="lists_1080p", kind="lists", n=700_001, width=1920, height=1080, tile_x=16, tile_y=16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _image(rng, lo, hi):
    width = _log(rng, lo, hi)
    return width, max(16, int(width * rng.uniform(0.5, 0.8)))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "lidar", "rig", "render", "render", "raster", "raster", "colours",
                       "lists"])
    if kind == "frame":
        w, h = _image(rng, 256, 1920)
        scene = rng.choice(["box", "wide", "wide", "frustum"])
        most = {"box": 100_000, "wide": 1_500_000, "frustum": 500_000}[scene]
        return dict(kind=kind, scene=scene, n=_log(rng, 10_000, most), width=w, height=h, degree=rng.randint(0, 3),
                    train=rng.random() < 0.7)
    if kind == "lidar":
        return dict(kind=kind, n=_log(rng, 100_000, 3_000_000), width=_log(rng, 512, 2048),
                    height=rng.choice([32, 64, 80, 128]), train=rng.random() < 0.7)
    if kind == "rig":
        w, h = _image(rng, 480, 1600)
        return dict(kind=kind, n=_log(rng, 200_000, 3_000_000), width=w, height=h, cameras=rng.randint(2, 6),
                    train=rng.random() < 0.7)
    if kind == "render":
        w, h = _image(rng, 320, 1600)
        shutter = rng.random() < 0.6
        return dict(kind=kind, lens=rng.choice(["pinhole", "distorted", "fisheye"]), n=_log(rng, 20_000, 600_000),
                    width=w, height=h, shutter=shutter, motion=shutter and rng.random() < 0.5,
                    train=rng.random() < 0.7)
    if kind == "raster":
        w, h = _image(rng, 256, 960)
        tx, ty = rng.choice([(16, 16), (16, 16), (32, 8), (8, 8), (16, 8)])
        return dict(kind=kind, n=_log(rng, 5_000, 60_000), width=w, height=h,
                    channels=rng.choice([1, 2, 3, 3, 4, 8, 16, 32]), tile_x=tx, tile_y=ty,
                    motion=rng.random() < 0.3, ray_grads=rng.random() < 0.3)
    if kind == "colours":
        return dict(kind=kind, n=_log(rng, 10_000, 2_000_000), degree=rng.randint(0, 4), layout_3kn=rng.random() < 0.5,
                    dc=rng.random() < 0.3, masked=rng.random() < 0.3)
    w, h = _image(rng, 320, 1920)
    tx, ty = rng.choice([(16, 16), (8, 8), (32, 8)])
    return dict(kind=kind, n=_log(rng, 10_000, 1_000_000), width=w, height=h, tile_x=tx, tile_y=ty)


# ------------------------------------------------------------------------------------------- scenes
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _bands(degree):
    return (degree + 1) ** 2


def _view_scene(case, g):
    """Gaussians in front of a pinhole camera at the origin looking along z, and the camera's focal lengths
    in pixels. ``box``: a shallow box; ``wide``: directions well past the image on every side; ``frustum``:
    directions that fill the image."""
    n, w, h = case["n"], case["width"], case["height"]
    u = _rand(g, n, 3)
    if case.get("scene") == "box":
        means = torch.stack([-5.0 + 10.0 * u[:, 0], -2.0 + 4.0 * u[:, 1], 2.0 + 18.0 * u[:, 2]], -1)
        f, spread = 1.0 * w, 0.5
    else:
        z = torch.exp(math.log(2.0) + math.log(40.0) * u[:, 2])
        f = 0.9 * w
        sx, sy = (0.5 * w / f, 0.5 * h / f) if case.get("scene", "frustum") == "frustum" else (1.2, 1.2)
        means = torch.stack([(2 * u[:, 0] - 1) * sx * z, (2 * u[:, 1] - 1) * sy * z, z], -1)
        spread = 0.7
    log_s = -3.0 + spread * _randn(g, n, 3)
    quats = torch.nn.functional.normalize(_randn(g, n, 4), dim=1)
    logits = 1.5 * _randn(g, n)
    return means, log_s, quats, logits, f


def _sh(g, n, degree):
    dc = 0.3 * _randn(g, n, 1, 3)
    return torch.cat([dc, 0.05 * _randn(g, n, _bands(degree) - 1, 3)], 1).contiguous()


def _image_grads(g, lead, channels):
    return (1e-3 * _randn(g, *lead, channels), 1e-3 * _randn(g, *lead), 1e-3 * _randn(g, *lead))


def _frame_scene(case, seed):
    from xsimgs_amd import synthetic as S

    g = _gen(seed)
    kind, n, w, h = case["kind"], case["n"], case["width"], case["height"]
    tile, sh, colors, degree, phm = (16, 16), None, None, 0, False
    if kind == "frame":
        means, log_s, quats, logits, f = _view_scene(case, g)
        degree = case["degree"]
        sh = _sh(g, n, degree)
        cams = [S.pinhole(w, h, f, f, w / 2, h / 2)]
    elif kind == "lidar":
        u = _rand(g, n, 3)
        r = torch.exp(math.log(120.0) * u[:, 0])
        az = 2.0 * math.pi * u[:, 1]
        means = torch.stack([r * torch.cos(az), r * torch.sin(az), -2.0 + 8.0 * u[:, 2]], -1)
        log_s = -2.5 + 0.7 * _randn(g, n, 3)
        quats = torch.nn.functional.normalize(_randn(g, n, 4), dim=1)
        logits = 1.5 * _randn(g, n)
        colors = torch.stack([_rand(g, n), _randn(g, n)], -1)
        _, beam_v, limits = S.lidar_beams(h)
        cams = [S.CameraSpec("lidar", w, h, [1.0, 0.0, 0.0, 0.0], [0.0, 0.0, 0.0], limits, beam_v=beam_v)]
        tile, phm = (32, 8), True
    else:
        blobs = 2000
        cu = _rand(g, blobs, 3)
        cr, caz = 5.0 + 55.0 * cu[:, 0], 2.0 * math.pi * cu[:, 1]
        centres = torch.stack([cr * torch.cos(caz), cr * torch.sin(caz), -2.0 + 8.0 * cu[:, 2]], -1)
        pick = torch.randint(0, blobs, (n,), generator=g, device=DEV)
        means = centres[pick] + 1.5 * _randn(g, n, 3)
        log_s = -3.0 + 0.7 * _randn(g, n, 3)
        quats = torch.nn.functional.normalize(_randn(g, n, 4), dim=1)
        logits = 1.0 + _randn(g, n)
        degree = 3
        sh = _sh(g, n, degree)
        cams = S.rig_cameras(width=w, height=h, f=0.7875 * w, n_cams=case["cameras"])
    sc = S.Scene(kind, means, log_s, quats, logits, sh, degree, colors, cams, tile, case["train"], use_phm=phm)
    lead = (case["cameras"], h, w) if kind == "rig" else (h, w)
    return sc, _image_grads(g, lead, 3 if sh is not None else 2)


_LENS = {"distorted": [-0.28, 0.07, 1e-3, -5e-4, 0.01, 0.02, -0.004, 0.001], "fisheye": [0.03, -0.005, 0.001, -1e-4]}


def _render_inputs(case, seed):
    from xsimgs_amd import frame, synthetic as S

    g = _gen(seed)
    n, w, h, lens = case["n"], case["width"], case["height"], case["lens"]
    means, log_s, quats, logits, f = _view_scene(dict(case, scene="frustum"), g)
    spec = S.pinhole(w, h, f, f, w / 2, h / 2)
    if lens == "fisheye":
        spec = S.CameraSpec(lens, w, h, spec.q, spec.t, [0.5, 0.5 * w / h, 0.5, 0.5], dist=_LENS[lens])
    elif lens == "distorted":
        spec = S.CameraSpec(lens, w, h, spec.q, spec.t, spec.impl, dist=_LENS[lens], max_radius=1.5)
    if case["shutter"]:
        spec.v, spec.w = [1.5, 0.2, -0.4], [0.03, -0.05, 0.1]
        spec.rolling, spec.trigger_time, spec.pose_time = [0.0, 0.04], 0.0, 0.02
    leaves = dict(points=means, log_s=log_s, rotation=quats, logits=logits, colors=_rand(g, n, 3))
    if case["motion"]:
        leaves["velocity"] = 0.8 * _randn(g, n, 3)
    leaves = {k: v.contiguous().requires_grad_(case["train"]) for k, v in leaves.items()}
    return frame.make_camera(spec, torch.device(DEV)), leaves, _image_grads(g, (h, w), 3)


def _raster_inputs(case, seed):
    """The compositor's inputs: Gaussians, rays and the tile lists of a splat of each Gaussian."""
    g = _gen(seed)
    n, w, h, ch = case["n"], case["width"], case["height"], case["channels"]
    means, log_s, quats, logits, f = _view_scene(dict(case, scene="frustum"), g)
    scales, opac = torch.exp(log_s), torch.sigmoid(logits)
    ray_o, ray_d = _pinhole_rays(w, h, f, torch.float32)
    velocity = times = None
    if case["motion"]:  # a moving camera and moving Gaussians, a row at a time
        velocity = 0.5 * _randn(g, n, 3)
        times = (torch.arange(h, device=DEV) / h - 0.5).view(h, 1, 1).expand(h, w, 1) * 0.04
        times = times.contiguous()
        ray_o = (ray_o + times * torch.tensor([1.5, 0.2, -0.4], device=DEV)).contiguous()
    m2, radii, depth = _splat(means, scales, quats, opac, w, h, f)
    offsets, flat, _ = _lists(m2, radii, depth, w, h, case["tile_x"], case["tile_y"])
    colors = _rand(g, n, ch)
    return dict(means=means.contiguous(), quats=quats, scales=scales, opac=opac, colors=colors, ray_o=ray_o,
                ray_d=ray_d, velocity=velocity, times=times, offsets=offsets, flat=flat,
                grads=_image_grads(g, (h, w), ch))


def _colour_inputs(case, seed):
    g = _gen(seed)
    n, k = case["n"], _bands(case["degree"])
    positions = 10.0 * _randn(g, n, 3) + torch.tensor([0.0, 0.0, 20.0], device=DEV)
    coeffs = _sh(g, n, case["degree"])
    dc = None
    if case["dc"] and k > 1:
        dc, coeffs = coeffs[:, :1].contiguous(), coeffs[:, 1:].contiguous()
    if case["layout_3kn"]:
        coeffs = coeffs.permute(2, 1, 0).contiguous()
        dc = dc.permute(2, 1, 0).contiguous() if dc is not None else None
    mask = torch.randint(-2**31, 2**31, ((n + 31) // 32,), generator=g, device=DEV).int() if case["masked"] else None
    return dict(coeffs=coeffs, dc=dc, positions=positions.contiguous(), mask=mask,
                origin=torch.tensor([0.5, -0.25, 1.0], device=DEV), grad=1e-3 * _randn(g, n, 3))


def _list_inputs(case, seed):
    """The case's own footprints on the image, in an order and at depths of the seed's (the lists then have
    one length for every seed)."""
    g = _gen(0)
    means, log_s, quats, logits, f = _view_scene(dict(case, scene="wide"), g)
    opac = torch.sigmoid(logits)
    m2, radii, _ = _splat(means, torch.exp(log_s), quats, opac, case["width"], case["height"], f)
    g = _gen(seed)
    order = torch.randperm(case["n"], generator=g, device=DEV)
    depth = torch.exp(math.log(2.0) + math.log(40.0) * _rand(g, case["n"]))
    return m2[order].contiguous(), radii[order].contiguous(), depth


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("frame", "lidar", "rig"):
        from xsimgs_amd import frame
        scene, grads = _frame_scene(case, seed)
        return dict(case=case, frame=frame.prepare(scene, DEV, requires_grad=case["train"]), grads=grads)
    if kind == "render":
        cam, leaves, grads = _render_inputs(case, seed)
        return dict(case=case, cam=cam, leaves=leaves, grads=grads)
    if kind == "raster":
        state = _raster_inputs(case, seed)
        keys = ["means", "quats", "scales", "opac", "colors"] + (["velocity", "times"] if case["motion"] else [])
        keys += ["ray_o", "ray_d"] if case["ray_grads"] else []
        for k in keys:
            state[k] = state[k].requires_grad_(True)
        return dict(state, case=case, leaves=keys)
    if kind == "colours":
        state = _colour_inputs(case, seed)
        leaves = [state[k].requires_grad_(True) for k in ("coeffs", "dc", "positions") if state[k] is not None]
        return dict(state, case=case, leaves=leaves)
    m2, radii, depth = _list_inputs(case, seed)
    return dict(case=case, means2d=m2, radii=radii, depth=depth)


# ---------------------------------------------------------------------------------------------- run
def run(state):
    case = state["case"]
    return {"frame": _run_frame, "lidar": _run_frame, "rig": _run_frame, "render": _run_render,
            "raster": _run_raster, "colours": _run_colours, "lists": _run_lists}[case["kind"]](case, state)


def _run_frame(case, state):
    from xsimgs_amd import frame

    st = state["frame"]
    call = frame.render_rig if case["kind"] == "rig" else frame.render_frame
    if not case["train"]:
        with torch.no_grad():
            out = call(st)
        return [out["rgb"], out["depth"], out["alpha"]]
    frame.zero_grads(st)
    out = call(st, backward=True, grads=state["grads"])
    return [out["rgb"], out["depth"], out["alpha"]] + [v for _, v in sorted(out["grads"].items()) if v is not None]


def _run_render(case, state):
    from xsimgs_amd.rendering import activate_gaussians, ut_gs_render

    x = state["leaves"]
    with torch.set_grad_enabled(case["train"]):
        scales, opac = activate_gaussians(x["log_s"], x["logits"])
        rgb, depth, alpha, meta = ut_gs_render(state["cam"], x["points"], scales, x["rotation"], opac, case["width"],
                                               case["height"], colors=x["colors"],
                                               points_velocity=x.get("velocity"))
    if not case["train"]:
        return [rgb, depth, alpha]
    grads = torch.autograd.grad([rgb, depth, alpha], list(x.values()), state["grads"])
    return [rgb, depth, alpha] + list(grads)


def _run_raster(case, state):
    from xsimgs_amd.rendering import ut_gs_dynamic_rasterize, ut_gs_rasterize

    s = state
    common = dict(positions=s["means"], rotation=s["quats"], scale=s["scales"], density=s["opac"], colors=s["colors"],
                  ray_o=s["ray_o"], ray_d=s["ray_d"], isect_offsets=s["offsets"], flatten_ids=s["flat"],
                  tile_size_x=case["tile_x"], tile_size_y=case["tile_y"])
    if case["motion"]:
        out = ut_gs_dynamic_rasterize(**common, velocity=s["velocity"], ray_time_delta=s["times"])
    else:
        out = ut_gs_rasterize(**common)
    return list(out) + list(torch.autograd.grad(out, [s[k] for k in s["leaves"]], s["grads"]))


def _run_colours(case, state):
    from xsimgs_amd.rendering import spherical_harmonics_fused

    s = state
    out = spherical_harmonics_fused(s["coeffs"], s["positions"], s["origin"], case["degree"], mask=s["mask"],
                                    layout_3kn=case["layout_3kn"], coeffs_dc=s["dc"])
    return [out] + list(torch.autograd.grad(out, s["leaves"], s["grad"]))


def _run_lists(case, state):
    from xsimgs_amd import _C

    w, h, tx, ty = case["width"], case["height"], case["tile_x"], case["tile_y"]
    per, keys, flat = _C.isect_regular_tiles(state["means2d"], state["radii"], state["depth"], w, h, tx, ty, sort=True)
    return [per, keys, flat, _C.isect_offset_encode(keys, -(-w // tx), -(-h // ty))]


# --------------------------------------------------------------------------- work and tolerances
def work(case):
    """Bytes: every input read once, every output written once; a Gaussian out of view costs its projection's
    inputs and, in training, its gradients. Operations: of the pixel-Gaussian pairs that are composited, at
    about 60 in a pass forward and 110 backward (nothing else comes near them)."""
    kind, n = case["kind"], case["n"]
    if kind == "colours":
        k, kept = _bands(case["degree"]), 0.5 if case["masked"] else 1.0
        return {"bytes": n * (12 + 12 + 12 + 12 + 12 * k * (1 + kept)), "flops": n * k * 20}
    if kind == "lists":
        return {"bytes": n * 24 + 12 * _entries(case), "flops": 0}
    pixels = case["width"] * case["height"] * case.get("cameras", 1)
    train = case.get("train", True)
    channels = {"lidar": 2, "raster": case.get("channels", 3)}.get(kind, 3)
    image = 4 * (channels + 2)
    per_gaussian = 44.0
    if kind in ("frame", "rig"):
        seen = 0.14 if case.get("scene") == "wide" else 1.0
        per_gaussian += 12 * _bands(case.get("degree", 3)) * seen
        grads = 44 + 12 * _bands(case.get("degree", 3))
    else:
        per_gaussian += 4 * channels + (12 if case.get("motion") else 0)
        grads = per_gaussian
    total = n * per_gaussian + pixels * image + (24 * pixels if kind == "raster" else 0)
    pairs = 66.0 * pixels * {"box": 0.2, "frustum": 0.8}.get(case.get("scene", "wide"), 1.0)
    flops = pairs * (55 + 2 * channels)
    if train:
        total += n * grads + pixels * image + (24 * pixels if case.get("ray_grads") else 0)
        flops += pairs * (110 + 4 * channels)
    return {"bytes": total, "flops": flops}


def _entries(case):
    return 12.4 * case["n"] * (case["width"] / 1920.0) ** 2 * 256 / (case["tile_x"] * case["tile_y"])


def tolerance(case):
    """Float32 throughout: about four times what the passes were measured to differ from ``exact`` by. Images:
    up to 6e-6, from single pixels where a float32 alpha or transmittance falls on the other side of its
    threshold (one such pixel is what ``max`` allows). Gradients: up to 1.9e-4, most of it from the pixels'
    remaining transmittance, which the backward takes from the float32 alpha image (a pixel that is nearly
    opaque keeps few digits of it); the tails belong to thin Gaussians, whose gradient is the small difference
    of large terms. A second pass, whose atomic sums run in another order, differs by 5e-7."""
    kind = case["kind"]
    if kind == "lists":
        return "exact"
    if kind == "colours":
        return {"rel": 1e-6, "max": 1e-4}
    if not case.get("train", True):
        return {"rel": 3e-5, "max": 0.2}
    return {"rel": 1e-3, "max": 0.5}


# ---------------------------------------------------------------------------------- plain torch
def _pinhole_rays(w, h, f, dtype):
    x = (torch.arange(w, device=DEV, dtype=dtype) + 0.5 - 0.5 * w) / f
    y = (torch.arange(h, device=DEV, dtype=dtype) + 0.5 - 0.5 * h) / f
    d = torch.stack([x.view(1, w).expand(h, w), y.view(h, 1).expand(h, w), torch.ones(h, w, device=DEV, dtype=dtype)], -1)
    return torch.zeros(h, w, 3, device=DEV, dtype=dtype), torch.nn.functional.normalize(d, dim=-1).contiguous()


def _rotation(q):
    w, x, y, z = torch.nn.functional.normalize(q, dim=1).unbind(1)
    return torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                        2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                        2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], 1).view(-1, 3, 3)


def _extent(opac):
    return torch.sqrt(2 * torch.log((opac * 255).clamp_min(1.0))).clamp_max(3.33)


def _splat(means, scales, quats, opac, w, h, f):
    """Image mean, radii (zero off screen) and depth of each Gaussian by its linearised projection."""
    x, y, z = means.unbind(1)
    r = _rotation(quats) * scales.unsqueeze(1)
    jx = f / z.unsqueeze(1) * (r[:, 0] - (x / z).unsqueeze(1) * r[:, 2])
    jy = f / z.unsqueeze(1) * (r[:, 1] - (y / z).unsqueeze(1) * r[:, 2])
    m2 = torch.stack([f * x / z + 0.5 * w, f * y / z + 0.5 * h], 1)
    radii = _extent(opac).unsqueeze(1) * torch.stack([jx.norm(dim=1), jy.norm(dim=1)], 1)
    size = torch.tensor([float(w), float(h)], device=DEV, dtype=m2.dtype)
    seen = ((m2 + radii >= 0) & (m2 - radii <= size)).all(1) & (opac >= 1 / 255)
    return m2, radii * seen.unsqueeze(1), z


def _project(means, scales, quats, opac, w, h, f):
    """Image mean, radii and depth by the unscented transform (alpha 0.1, beta 2, kappa 0) of a pinhole
    camera at the origin: seven sigma points, all of them within one image size of the image."""
    spread = 0.03
    d = (_rotation(quats) * scales.unsqueeze(1)).transpose(1, 2) * math.sqrt(spread)
    pts = torch.cat([means.unsqueeze(1), means.unsqueeze(1) + d, means.unsqueeze(1) - d], 1)
    u = f / w * pts[..., 0] / pts[..., 2] + 0.5
    v = f / h * pts[..., 1] / pts[..., 2] + 0.5
    ok = ((pts[..., 2] > 0) & (u >= -1) & (u <= 2) & (v >= -1) & (v <= 2)).all(1)
    p = torch.stack([u * w, v * h], -1)
    m2 = (spread - 3) / spread * p[:, 0] + p[:, 1:].sum(1) / (2 * spread)
    e = p - m2.unsqueeze(1)
    wc = torch.full((7,), 1 / (2 * spread), device=DEV, dtype=p.dtype)
    wc[0] = (spread - 3) / spread + 1 - 0.01 + 2
    cov = (wc.view(1, 7, 1) * e * e).sum(1)
    cxy = (wc.view(1, 7) * e[..., 0] * e[..., 1]).sum(1)
    ok = ok & (cov[:, 0] * cov[:, 1] - cxy * cxy > 0) & (cov >= 0).all(1) & (opac >= 1 / 255)
    radii = _extent(opac).unsqueeze(1) * torch.sqrt(cov.clamp_min(0))
    size = torch.tensor([float(w), float(h)], device=DEV, dtype=p.dtype)
    ok = ok & ((m2 + radii >= 0) & (m2 - radii <= size)).all(1)
    return m2, radii * ok.unsqueeze(1), means[:, 2]


def _lists(m2, radii, depth, w, h, tx, ty):
    """Per tile, the Gaussians whose rectangle touches it in depth order: offsets, ids and their number."""
    nx, ny = -(-w // tx), -(-h // ty)
    size = torch.tensor([tx, ty], device=DEV, dtype=m2.dtype)
    most = torch.tensor([nx, ny], device=DEV)
    seen = (radii > 0).all(1)
    m2, radii = torch.where(seen[:, None], m2, 0.0), torch.where(seen[:, None], radii, 0.0)
    lo = torch.minimum(torch.floor((m2 - radii) / size).clamp_min(0).long(), most)
    hi = torch.minimum(torch.ceil((m2 + radii) / size).clamp_min(0).long(), most)
    span = (hi - lo) * seen.unsqueeze(1)
    count = span[:, 0] * span[:, 1]
    order = torch.argsort(depth, stable=True)
    c = count[order]
    ids = torch.repeat_interleave(order, c)
    k = torch.arange(ids.numel(), device=DEV) - torch.repeat_interleave(torch.cumsum(c, 0) - c, c)
    sx = span[ids, 0]
    row = torch.div(k, sx.clamp_min(1), rounding_mode="floor")
    tile = (lo[ids, 1] + row) * nx + lo[ids, 0] + (k - row * sx)
    tile, at = torch.sort(tile, stable=True)
    offsets = torch.searchsorted(tile, torch.arange(nx * ny, device=DEV))
    return offsets.int().view(ny, nx), ids[at].int(), ids.numel()


def _sh_colours(coeffs, positions, origin, degree):
    """Half plus real spherical harmonics up to degree 4 of the direction origin -> position; bands in dim 1."""
    x, y, z = torch.nn.functional.normalize(positions - origin, dim=1).unbind(1)
    xx, yy, zz = x * x, y * y, z * z
    b = [torch.full_like(x, 0.28209479177387814)]
    if degree > 0:
        c = 0.4886025119029199
        b += [-c * y, c * z, -c * x]
    if degree > 1:
        b += [1.0925484305920792 * x * y, -1.0925484305920792 * y * z, 0.31539156525252005 * (2 * zz - xx - yy),
              -1.0925484305920792 * x * z, 0.5462742152960396 * (xx - yy)]
    if degree > 2:
        b += [-0.5900435899266435 * y * (3 * xx - yy), 2.890611442640554 * x * y * z,
              -0.4570457994644658 * y * (4 * zz - xx - yy), 0.3731763325901154 * z * (2 * zz - 3 * xx - 3 * yy),
              -0.4570457994644658 * x * (4 * zz - xx - yy), 1.445305721320277 * z * (xx - yy),
              -0.5900435899266435 * x * (xx - 3 * yy)]
    if degree > 3:
        b += [2.5033429417967046 * x * y * (xx - yy), -1.7701307697799304 * y * z * (3 * xx - yy),
              0.9461746957575601 * x * y * (7 * zz - 1), -0.6690465435572892 * y * z * (7 * zz - 3),
              0.10578554691520431 * (zz * (35 * zz - 30) + 3), -0.6690465435572892 * x * z * (7 * zz - 3),
              0.47308734787878004 * (xx - yy) * (7 * zz - 1), -1.7701307697799304 * x * z * (xx - 3 * yy),
              0.6258357354491761 * (xx * (xx - 3 * yy) - yy * (3 * xx - yy))]
    return (torch.stack(b, 1).unsqueeze(2) * coeffs).sum(1) + 0.5


def _composite(means, quats, scales, opac, colors, ray_o, ray_d, offsets, flat, tx, ty, grads=None, velocity=None,
               times=None):
    """The images [rgb, depth, alpha] of the tile lists and, with the images' gradients, those of means, quats,
    scales, opacities, colours, velocities, times, ray origins and ray directions, by name; in float64. Tiles
    of similar length are evaluated together."""
    h, w = ray_o.shape[:2]
    ny, nx = offsets.shape
    ch, p = colors.shape[1], tx * ty
    pad = (0, 0, 0, nx * tx - w, 0, ny * ty - h)

    def tiles_of(t):  # [h, w, c] -> [tiles, pixels, c]
        t = torch.nn.functional.pad(t.double(), pad)
        return t.view(ny, ty, nx, tx, -1).permute(0, 2, 1, 3, 4).reshape(ny * nx, p, -1)

    def image_of(t):
        return t.view(ny, nx, ty, tx, -1).permute(0, 2, 1, 3, 4).reshape(ny * ty, nx * tx, -1)[:h, :w].contiguous()

    q, s = quats.detach().double().requires_grad_(True), scales.detach().double().requires_grad_(True)
    rows = _rotation(q).transpose(1, 2) / s.unsqueeze(2)
    m, mu, op, col = rows.detach().contiguous(), means.detach().double(), opac.detach().double(), colors.detach().double()
    vel = velocity.detach().double() if velocity is not None else None
    ro, rd = tiles_of(ray_o.detach()), tiles_of(ray_d.detach())
    rt = tiles_of(times.detach()) if times is not None else None
    one_origin = bool((ray_o == ray_o[0, 0]).all())
    inside = tiles_of(torch.ones(h, w, 1, device=DEV))[..., 0] > 0
    rd[~inside] = 1.0  # a padding pixel's ray is of no account, but not zero
    starts = offsets.view(-1).long()
    counts = torch.diff(starts, append=torch.tensor([flat.numel()], device=DEV))
    order = torch.argsort(counts, descending=True)
    sizes = counts[order].tolist()
    out = torch.zeros(ny * nx, p, ch + 2, device=DEV, dtype=torch.float64)
    acc = {}
    if grads is not None:
        vi = [tiles_of(t.view(h, w, -1)) for t in grads]
        acc = {k: torch.zeros(mu.shape[0], c, device=DEV, dtype=torch.float64)
               for k, c in (("m", 9), ("means", 3), ("opac", 1), ("colors", ch), ("velocity", 3))}
        acc.update({k: torch.zeros(ny * nx, p, c, device=DEV, dtype=torch.float64)
                    for k, c in (("ray_o", 3), ("ray_d", 3), ("times", 1))})
    i = 0
    while i < len(sizes) and sizes[i] > 0:
        gn = sizes[i]
        t = order[i:i + max(1, (12 << 20) // (gn * p))]
        i += t.numel()
        k = torch.arange(gn, device=DEV)
        live = (k < counts[t].unsqueeze(1)).unsqueeze(2) & inside[t].unsqueeze(1)
        ids = flat[(starts[t].unsqueeze(1) + k).clamp_max(flat.numel() - 1)].long()
        mm, mui, opi, ci = m[ids], mu[ids], op[ids].unsqueeze(2), col[ids]
        nt = t.numel()

        def mapped(v):  # M v for the pixels' vectors [tiles, pixels, 3] -> [tiles, gaussians, 3, pixels]
            return (mm.view(nt, gn * 3, 3) @ v.transpose(1, 2)).view(nt, gn, 3, -1)

        grd = mapped(rd[t])
        gro = mapped(ro[t][:, :1] if one_origin else ro[t]) - (mm @ mui.unsqueeze(3))
        if vel is not None:
            mv = mm @ vel[ids].unsqueeze(3)
            gro = gro - mv * rt[t].view(nt, 1, 1, p)
        dd = (grd * grd).sum(2)
        gro = gro.expand_as(grd)
        c = torch.linalg.cross(grd, gro, dim=2)
        cc, od = (c * c).sum(2), (grd * gro).sum(2)
        vis = torch.exp(-0.5 * cc / dd)
        raw = opi * vis
        a = torch.where(live & (raw >= 1 / 255), raw.clamp_max(0.999), 0.0)
        after = torch.cumprod(1 - a, 1)
        taken = (a > 0) & (after > 1e-4)
        a = torch.where(taken, a, 0.0)
        after = torch.cumprod(1 - a, 1)
        wgt = a * torch.cat([torch.ones_like(after[:, :1]), after[:, :-1]], 1)
        hit = -od / dd
        last = after[:, -1]
        out[t] = torch.cat([wgt.transpose(1, 2) @ ci, (wgt * hit).sum(1).unsqueeze(2), (1 - last).unsqueeze(2)], 2)
        if grads is None:
            continue
        v_rgb, v_d, v_a = vi[0][t], vi[1][t].view(nt, 1, p), vi[2][t].view(nt, p)
        ab = torch.where(taken, raw.clamp_max(0.99), 0.0)
        trans = last.unsqueeze(1) / torch.flip(torch.cumprod(torch.flip(1 - ab, [1]), 1), [1])
        fac = ab * trans
        u = ci @ v_rgb.transpose(1, 2) + hit * v_d
        fu = fac * u
        behind = torch.flip(torch.cumsum(torch.flip(fu, [1]), 1), [1]) - fu
        v_alpha = trans * u - (behind - (last * v_a).unsqueeze(1)) / (1 - ab)
        geo = taken & (raw <= 0.99)
        v_alpha, v_hit = torch.where(geo, v_alpha, 0.0), torch.where(geo, v_d * fac, 0.0)
        amount = raw * v_alpha
        v_c = -(amount / dd).unsqueeze(2) * c
        v_dd = 0.5 * amount * cc / (dd * dd) + v_hit * od / (dd * dd)
        v_grd = torch.linalg.cross(gro, v_c, dim=2) + 2 * grd * v_dd.unsqueeze(2) - gro * (v_hit / dd).unsqueeze(2)
        v_gro = torch.linalg.cross(v_c, grd, dim=2) - grd * (v_hit / dd).unsqueeze(2)
        total = v_gro.sum(3)
        v_m = (v_grd.reshape(nt, gn * 3, p) @ rd[t]).view(nt, gn, 3, 3)
        v_m = v_m + (v_gro.reshape(nt, gn * 3, p) @ ro[t]).view(nt, gn, 3, 3) - total.unsqueeze(3) * mui.unsqueeze(2)
        if vel is not None:
            timed = (v_gro * rt[t].view(nt, 1, 1, p)).sum(3)
            v_m = v_m - timed.unsqueeze(3) * vel[ids].unsqueeze(2)
            acc["velocity"].index_add_(0, ids.view(-1), -(timed.unsqueeze(2) @ mm).view(-1, 3))
            acc["times"][t] = -(mv * v_gro).sum((1, 2)).unsqueeze(2)
        acc["m"].index_add_(0, ids.view(-1), v_m.view(-1, 9))
        acc["means"].index_add_(0, ids.view(-1), -(total.unsqueeze(2) @ mm).view(-1, 3))
        acc["opac"].index_add_(0, ids.view(-1), (vis * v_alpha).sum(2).view(-1, 1))
        acc["colors"].index_add_(0, ids.view(-1), (fac @ v_rgb).view(-1, ch))
        flat_m = mm.reshape(nt, gn * 3, 3)
        acc["ray_o"][t] = v_gro.reshape(nt, gn * 3, p).transpose(1, 2) @ flat_m
        acc["ray_d"][t] = v_grd.reshape(nt, gn * 3, p).transpose(1, 2) @ flat_m
    img = image_of(out)
    images = [img[..., :ch].contiguous(), img[..., ch].contiguous(), img[..., ch + 1].contiguous()]
    if grads is None:
        return images, None
    for k in ("ray_o", "ray_d", "times"):
        acc[k] = image_of(acc[k])
    acc["quats"], acc["scales"] = torch.autograd.grad(rows, [q, s], acc.pop("m").view(-1, 3, 3))
    acc["opac"] = acc["opac"].view(-1)
    return images, acc


_MOST_PAIRS = 5e9  # about twenty seconds of float64


def exact(case, seed):
    kind = case["kind"]
    if kind == "colours":
        return _exact_colours(case, seed)
    if kind == "raster":
        x = _raster_inputs(case, seed)
        if x["flat"].numel() * case["tile_x"] * case["tile_y"] > _MOST_PAIRS:
            return None
        images, acc = _composite(x["means"], x["quats"], x["scales"], x["opac"], x["colors"], x["ray_o"], x["ray_d"],
                                 x["offsets"], x["flat"], case["tile_x"], case["tile_y"], x["grads"], x["velocity"],
                                 x["times"])
        keys = ["means", "quats", "scales", "opac", "colors"] + (["velocity", "times"] if case["motion"] else [])
        keys += ["ray_o", "ray_d"] if case["ray_grads"] else []
        return images + [acc[k] for k in keys]
    if kind == "frame":
        return _exact_frame(case, seed)
    return None  # the lists of the other cameras' projections have no plain restatement here, lists no rounding


def _exact_colours(case, seed):
    x = _colour_inputs(case, seed)
    k, n = _bands(case["degree"]), case["n"]
    coeffs = x["coeffs"].detach().double().requires_grad_(True)
    dc = x["dc"].detach().double().requires_grad_(True) if x["dc"] is not None else None
    pos = x["positions"].double().requires_grad_(True)
    c, d = (coeffs, dc) if not case["layout_3kn"] else (coeffs.permute(2, 1, 0), dc.permute(2, 1, 0) if dc is not None else None)
    out = _sh_colours(torch.cat([d, c], 1) if d is not None else c, pos, x["origin"].double(), case["degree"])
    if x["mask"] is not None:
        i = torch.arange(n, device=DEV)
        out = out * ((x["mask"][i // 32] >> (i % 32)) & 1).double().unsqueeze(1)
    leaves = [t for t in (coeffs, dc, pos) if t is not None]
    grads = torch.autograd.grad(out, leaves, x["grad"].double(), allow_unused=True)
    return [out.detach()] + [torch.zeros_like(t) if g is None else g for t, g in zip(leaves, grads)]


def _exact_frame(case, seed):
    sc, grads = _frame_scene(case, seed)
    w, h, (tx, ty) = case["width"], case["height"], sc.tile_size
    f = sc.cameras[0].impl[0] * w
    means, quats = sc.means.double(), sc.quats.double()
    scales, opac = torch.exp(sc.log_scales.double()), torch.sigmoid(sc.opacity_logits.double())
    m2, radii, depth = _project(means, scales, quats, opac, w, h, f)
    offsets, flat, entries = _lists(m2, radii, depth, w, h, tx, ty)
    if entries * tx * ty > _MOST_PAIRS:
        return None
    seen = torch.unique(flat.long())  # the rest have no colour to compute and exact zero gradients
    at = torch.zeros(case["n"], dtype=torch.long, device=DEV)
    at[seen] = torch.arange(seen.numel(), device=DEV)
    sh = sc.sh_coeffs[seen].double().requires_grad_(True)
    pos = means[seen].requires_grad_(True)
    colors = _sh_colours(sh, pos, torch.zeros(3, device=DEV, dtype=torch.float64), case["degree"])
    ray_o, ray_d = _pinhole_rays(w, h, f, torch.float64)
    images, acc = _composite(pos, quats[seen], scales[seen], opac[seen], colors, ray_o, ray_d, offsets,
                             at[flat.long()], tx, ty, grads if case["train"] else None)
    if acc is None:
        return images
    v_sh, v_pos = torch.autograd.grad(colors, [sh, pos], acc["colors"], allow_unused=True)
    v_pos = torch.zeros_like(pos) if v_pos is None else v_pos

    def whole(v, shape):
        full = torch.zeros(shape, device=DEV, dtype=torch.float64)
        full[seen] = v
        return full

    n = case["n"]
    return images + [whole(acc["scales"] * scales[seen], (n, 3)), whole(acc["means"] + v_pos, (n, 3)),
                     whole(acc["opac"] * opac[seen] * (1 - opac[seen]), (n,)), whole(acc["quats"], (n, 4)),
                     whole(v_sh, tuple(sc.sh_coeffs.shape))]
