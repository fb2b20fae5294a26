"""The compositor's edge inputs against the float64 oracle: grids larger than the image, pixels without a ray,
tiles of very wide rays, flat Gaussians seen from moving origins, Gaussians whose turn is a near tie, and
Gaussians at the camera, Gaussians of no or infinite extent or that are no numbers, and
the launches whose LDS is sized for small workgroups.

Every tile lists the same Gaussians in depth order. Bounds are the suite's: 1e-4 absolute on the renders of all
but one pixel in ten thousand, 1e-3 of an array's norm on gradients.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from xsimgs_amd import _C
from tests._util import np_

pytestmark = pytest.mark.gpu


def _scene(W, H, tile, grid=None, n=150, cdim=3, moving=False, dynamic=False, seed=0, f=0.9):
    g = np.random.default_rng(seed)
    z = np.sort(g.uniform(3.0, 30.0, n))
    f = f * W
    x, y = (np.arange(W) + 0.5 - W / 2) / f, (np.arange(H) + 0.5 - H / 2) / f
    means = np.stack([g.uniform(-0.55, 0.55, n) * W / f * z, g.uniform(-0.55, 0.55, n) * H / f * z, z], -1)
    rd = np.stack([np.broadcast_to(x, (H, W)), np.broadcast_to(y[:, None], (H, W)), np.ones((H, W))], -1)
    rd /= np.linalg.norm(rd, axis=-1, keepdims=True)
    rows = (np.arange(H) / H)[:, None, None]
    ro = np.zeros((H, W, 3)) + [0.1, -0.2, 0.05] + (rows * [0.05, 0.0, -0.02] if moving or dynamic else 0.0)
    nty, ntx = grid or (-(-H // tile[1]), -(-W // tile[0]))
    s = dict(means=means, quats=g.normal(0, 1, (n, 4)),
             scales=np.exp(g.normal(np.log(0.12), 0.5, (n, 3))) * z[:, None] / 10 * W / f, colors=g.normal(0, 1, (n, cdim)),
             opac=g.uniform(0.02, 0.98, n), ro=ro, rd=rd)
    if dynamic:
        s.update(vel=0.5 * g.normal(0, 1, (n, 3)), rt=np.broadcast_to(rows[..., 0] * 0.04, (H, W)))
    s = {k: np.ascontiguousarray(a, np.float32) for k, a in s.items()}
    s.update(offsets=(np.arange(ntx * nty, dtype=np.int32) * n).reshape(nty, ntx),
             flat=np.tile(np.arange(n, dtype=np.int32), ntx * nty), tile=tile, size=(W, H))
    return s


def _forward(s, counts=None):
    T = {k: torch.from_numpy(a).cuda() for k, a in s.items() if isinstance(a, np.ndarray)}
    work = torch.full((s["offsets"].size,), -7, dtype=torch.int32, device="cuda")
    tail = (*s["size"], *s["tile"], T["ro"], T["rd"])
    kw = dict(tile_work=work, pair_counts=counts)
    if "vel" in s:
        out = _C.rasterize_eval3d_dynamic_fwd(T["means"], T["vel"], T["quats"], T["scales"], T["colors"].unsqueeze(0),
                                              T["opac"].view(1, -1), *tail, T["rt"], T["offsets"], T["flat"], **kw)
    else:
        out = _C.rasterize_eval3d_fwd(T["means"], T["quats"], T["scales"], T["colors"].unsqueeze(0),
                                      T["opac"].view(1, -1), *tail, T["offsets"], T["flat"], **kw)
    return out, work, T


def _backward(s, out, work, T, v, **kw):
    V = [torch.from_numpy(a).cuda() for a in v]
    tail = (*s["tile"], T["offsets"], T["flat"], out[2], out[3], *V)
    if "vel" in s:
        got = _C.rasterize_eval3d_dynamic_bwd(T["means"], T["vel"], T["scales"], T["quats"], T["opac"], T["colors"],
                                              T["ro"], T["rd"], T["rt"], *tail, tile_work=work, **kw)
        names = ["v_means", "v_velocity", "v_quats", "v_scales", "v_opacity", "v_colors", "v_ray_o", "v_ray_d",
                 "v_time_delta"]
    else:
        got = _C.rasterize_eval3d_bwd(T["means"], T["scales"], T["quats"], T["opac"], T["colors"], T["ro"], T["rd"],
                                      *tail, tile_work=work, **kw)
        names = ["v_means", "v_quats", "v_scales", "v_opacity", "v_colors", "v_ray_o", "v_ray_d"]
    return {k: np_(x) for k, x in zip(names, got) if x is not None}


def _oracle_fwd(s):
    return O.eval3d_fwd(s["means"], s["quats"], s["scales"], s["colors"], s["opac"], s["ro"], s["rd"], s["offsets"],
                        s["flat"], *s["tile"], velocity=s.get("vel"), ray_time_delta=s.get("rt"), prec="f64")


def _oracle_bwd(s, alpha, last, v, tiles=None):
    return O.eval3d_bwd(s["means"], s["quats"], s["scales"], s["colors"], s["opac"], s["ro"], s["rd"], s["offsets"],
                        s["flat"], alpha, last, *v, *s["tile"], velocity=s.get("vel"), ray_time_delta=s.get("rt"),
                        prec="f64", tiles=tiles)


def _check_images(out, ref, where, depth=True):
    for k, (got, want) in enumerate(zip(out[:3], ref[:3])):
        if k == 1 and not depth:
            continue
        bad = ~(np.abs(np_(got)[where] - want[where]) <= 1e-4 * np.maximum(1.0, np.abs(want[where])))
        assert bad.mean() <= 1e-4, (k, bad.mean())
    assert (np_(out[3])[where] != ref[3][where]).mean() <= 1e-4


def _check_grads(got, ref, where=None):
    for name, x in got.items():
        want = ref[name]
        if where is not None and x.shape[:2] == where.shape:
            x, want = x[where], want[where]
        err = np.linalg.norm((x - want).reshape(-1))
        assert err <= 1e-3 * np.linalg.norm(want) + 1e-12, (name, err, np.linalg.norm(want))


def _image_grads(W, H, cdim, seed=7):
    g = np.random.default_rng(seed)
    return [g.normal(0, 1e-3, shape).astype(np.float32) for shape in ((H, W, cdim), (H, W), (H, W))]


@pytest.mark.parametrize("dynamic", [False, True])
@pytest.mark.parametrize("size,tile,grid", [((40, 33), (16, 16), (4, 5)), ((64, 48), (32, 32), (3, 3)),
                                            ((31, 17), (8, 8), (3, 9)), ((20, 70), (12, 10), (12, 2))])
def test_grid_larger_than_image(size, tile, grid, dynamic):
    """Tiles past the image hold no pixel: their lists are not read, and the rest is as in the exact grid."""
    W, H = size
    s = _scene(W, H, tile, grid, dynamic=dynamic)
    out, work, T = _forward(s)
    _check_images(out, _oracle_fwd(s), np.ones((H, W), bool))
    rows, cols = np.meshgrid(np.arange(grid[0]) * tile[1], np.arange(grid[1]) * tile[0], indexing="ij")
    assert np.array_equal(np_(work).reshape(grid) > 0, (rows < H) & (cols < W))
    assert (np_(work) >= 0).all()
    v = _image_grads(W, H, 3)
    ref = _oracle_bwd(s, np_(out[2]), np_(out[3]), v)
    for kw in (dict(ray_grads=True), dict(ray_grads=False, pixels_per_lane=2), dict(ray_grads=False, pixels_per_lane=4)):
        _check_grads(_backward(s, out, work, T, v, **kw), ref)


def test_grid_larger_than_images_batched():
    """The same with three cameras: no camera's tiles past its image take another's rays."""
    W, H, tile, grid, n = 40, 33, (16, 16), (4, 4), 150
    scenes = [_scene(W, H, tile, grid, n=n, seed=3) for _ in range(3)]
    for c, s in enumerate(scenes):
        s["ro"] = s["ro"] + np.float32([0.1 * c, 0.0, 0.0])
    cat = lambda k: torch.from_numpy(np.stack([s[k] for s in scenes])).cuda()
    T = {k: torch.from_numpy(a).cuda() for k, a in scenes[0].items() if isinstance(a, np.ndarray)}
    per = grid[0] * grid[1] * n
    offsets = torch.from_numpy(np.stack([s["offsets"] + c * per for c, s in enumerate(scenes)])).cuda()
    flat = torch.from_numpy(np.concatenate([s["flat"] + c * n for c, s in enumerate(scenes)])).cuda()
    out = _C.rasterize_eval3d_fwd_batched(T["means"], T["quats"], T["scales"], T["colors"], T["opac"], W, H, *tile,
                                          cat("ro"), cat("rd"), offsets, flat)
    v = [_image_grads(W, H, 3, seed=c) for c in range(3)]
    V = [torch.from_numpy(np.stack(a)).cuda() for a in zip(*v)]
    got = _C.rasterize_eval3d_bwd_batched(T["means"], T["scales"], T["quats"], T["opac"], T["colors"], cat("ro"),
                                          cat("rd"), *tile, offsets, flat, out[2], out[3], *V, ray_grads=True)
    total = {}
    for c, s in enumerate(scenes):
        ref = list(_oracle_fwd(s))
        last = np_(out[3][c]) - c * per
        last[np_(out[2][c]) == 0.0] = 0  # (a pixel without any Gaussian reports 0)
        _check_images([out[0][c], out[1][c], out[2][c], last], ref, np.ones((H, W), bool))
        one = _oracle_bwd(s, np_(out[2][c]), last, v[c])
        _check_grads(dict(v_ray_o=np_(got[5][c]), v_ray_d=np_(got[6][c])), one)
        for k in ("v_means", "v_quats", "v_scales", "v_opacity", "v_colors"):
            total[k] = total.get(k, 0.0) + one[k]
    _check_grads({k: np_(x) for k, x in zip(("v_means", "v_quats", "v_scales", "v_opacity", "v_colors"), got)}, total)


def _spoil(s, where, kind):
    """Takes the rays of some pixels away: the middle one of every tile, more than a
    strip of 64, a whole tile."""
    W, H = s["size"]
    tw, th = s["tile"]
    j, i = np.meshgrid(np.arange(W), np.arange(H))
    if where == "middle":
        bad = (j % tw == min(tw // 2, W - 1)) & (i % th == min(th // 2, H - 1))
    elif where == "strip":
        bad = i % th < min(64 // tw + 1, th // 2)
    else:
        bad = (j // tw == 1) & (i // th == 1)
    if kind == "time":
        s["rt"] = s["rt"].copy()
        s["rt"][bad] = np.nan
    else:
        s["rd"][bad] = dict(zero=0.0, nan=np.nan)[kind]
    return bad


@pytest.mark.parametrize("tile", [(16, 16), (32, 32), (8, 8)])
@pytest.mark.parametrize("where", ["middle", "strip", "tile"])
@pytest.mark.parametrize("kind,moving,dynamic", [("zero", False, False), ("nan", False, False), ("zero", True, False),
                                                 ("nan", False, True), ("time", False, True), ("zero", False, True)])
def test_pixels_without_a_ray(kind, moving, dynamic, where, tile):
    """A zero direction meets every Gaussian at its full opacity, a NaN one at 0.999, and neither changes another
    pixel. (Their depths are not compared, 0 / 0 in the oracle; gradients are those of the other pixels.)"""
    W, H = 97, 81
    s = _scene(W, H, tile, moving=moving, dynamic=dynamic)
    bad = _spoil(s, where, kind)
    s["opac"][::7] = 0.002  # (below the threshold, but not at 0.999)
    out, work, T = _forward(s)
    ref = _oracle_fwd(s)
    _check_images(out, ref, ~bad)
    _check_images(out, ref, bad, depth=False)
    if kind != "zero":
        return
    v = _image_grads(W, H, 3)
    last = np_(out[3]).copy()
    last[bad] = -1
    for a in v:
        a[bad] = 0.0
    want = _oracle_bwd(s, np_(out[2]), last, v)
    for kw in (dict(ray_grads=True), dict(ray_grads=False, pixels_per_lane=2), dict(ray_grads=False, pixels_per_lane=4)):
        _check_grads(_backward(s, out, work, T, v, **kw), want, ~bad)


def _pair_counts(s):
    """Evaluated pairs of the forward and of the backward (ray gradients, two and four pixels per lane)."""
    n = [torch.zeros(2, dtype=torch.int64, device="cuda") for _ in range(4)]
    out, work, T = _forward(s, n[0])
    v = _image_grads(*s["size"], 3)
    for c, kw in zip(n[1:], (dict(ray_grads=True), dict(ray_grads=False, pixels_per_lane=2),
                             dict(ray_grads=False, pixels_per_lane=4))):
        _backward(s, out, work, T, v, pair_counts=c, **kw)
    return np.array([int(c[0]) for c in n])


@pytest.mark.parametrize("moving,dynamic", [(False, False), (True, False), (False, True)])
@pytest.mark.parametrize("where", ["middle", "corner"])
def test_a_pixel_without_a_ray_costs_its_strip(where, moving, dynamic):
    """One pixel of a 16x16 tile without a ray leaves the tile's other three strips of 64 pixels culled as before."""
    W, H = 96, 80
    s = _scene(W, H, (16, 16), moving=moving, dynamic=dynamic)
    clean = _pair_counts(s)
    if where == "middle":
        _spoil(s, "middle", "zero")
    else:
        s["rd"][::16, ::16] = 0.0
    most = clean + (W // 16) * (H // 16) * 64 * s["means"].shape[0]
    got = _pair_counts(s)
    print("evaluated", clean, got, "at most", most)
    assert (got <= most).all()


@pytest.mark.parametrize("size,tile,f", [((32, 32), (32, 32), 0.25), ((64, 32), (32, 32), 0.1), ((48, 16), (16, 16), 0.1)])
def test_wide_tiles(size, tile, f):
    """Tiles whose corners lie up to 80 degrees from their middle ray are culled too, and stay exact."""
    W, H = size
    s = _scene(W, H, tile, f=f)
    mid = s["rd"][min(tile[1] // 2, H - 1)][tile[0] // 2::tile[0]]
    angle = max(float(np.degrees(np.arccos((s["rd"][:tile[1], k * tile[0]:(k + 1) * tile[0]] @ m).min())))
                for k, m in enumerate(mid))
    assert 62.0 < angle < 84.0, angle
    out, work, T = _forward(s)
    _check_images(out, _oracle_fwd(s), np.ones((H, W), bool))
    v = _image_grads(W, H, 3)
    ref = _oracle_bwd(s, np_(out[2]), np_(out[3]), v)
    for kw in (dict(ray_grads=True), dict(ray_grads=False, pixels_per_lane=2), dict(ray_grads=False, pixels_per_lane=4)):
        _check_grads(_backward(s, out, work, T, v, **kw), ref)
    n = _pair_counts(s)
    print("evaluated", n, "of", W * H * s["means"].shape[0], "angle", angle)
    assert (n <= 0.5 * W * H * s["means"].shape[0]).all()


@pytest.mark.parametrize("dynamic", [False, True])
@pytest.mark.parametrize("flat", [1.0, 1e-2, 1e-3])
@pytest.mark.parametrize("tile", [(16, 16), (32, 32)])
def test_flat_gaussians_from_moving_origins(tile, flat, dynamic):
    """Origins that move by many times a flat Gaussian's thickness within a tile leave it culled by its other axes,
    and no pair is lost. Bound on the pairs: twice those of one origin, the ball that the motion adds to every
    Gaussian being smaller than its larger axes. The last ids and images are the oracle's but for the pairs that
    float32 cannot decide: its alpha is off by 17 ulp of |o - mu| / s_min there."""
    W, H = 96, 80
    s = _scene(W, H, tile, moving=True, dynamic=dynamic, n=300, seed=5)
    s["scales"][:, 0] = s["scales"].max(1) * flat
    still = dict(s, ro=np.ascontiguousarray(np.broadcast_to(s["ro"][H // 2, W // 2], s["ro"].shape)))
    if dynamic:
        still["rt"] = np.zeros_like(s["rt"])
    most = 2 * _pair_counts(still)
    n = _pair_counts(s)
    print("evaluated", n, "one origin", most // 2)
    assert (n <= most).all()
    out, work, T = _forward(s)
    ref = _oracle_fwd(s)
    share = 1e-4 if flat == 1.0 else 1e-2
    for got, want in zip((out[0], out[2]), (ref[0], ref[2])):
        assert (np.abs(np_(got) - want) > 1e-3).mean() <= share
    assert (np_(out[3]) != ref[3]).mean() <= share


def _quat_mul(a, b):
    w1, x1, y1, z1 = a.T
    w2, x2, y2, z2 = b.T
    return np.stack([w1 * w2 - x1 * x2 - y1 * y2 - z1 * z2, w1 * x2 + x1 * w2 + y1 * z2 - z1 * y2,
                     w1 * y2 - x1 * z2 + y1 * w2 + z1 * x2, w1 * z2 + x1 * y2 - y1 * x2 + z1 * w2], 1)


def test_turn_of_near_ties():
    """The largest components of M (o - mu) agree to about an ulp, so that rounding picks the axis of the turn: the
    backward turns the gradients back about the axis that it turned them by. Per Gaussian: 1e-3 of the gradient,
    the suite's bar, for those of at least a fifth of the usual size."""
    W = H = 64
    per, tile = 400, (16, 16)
    g = np.random.default_rng(2)
    s = _scene(W, H, tile, n=1, f=0.8)
    n = per * s["offsets"].size
    t = np.repeat(np.arange(s["offsets"].size), per)
    v = -s["rd"][t // 4 * 16 + g.integers(0, 16, n), t % 4 * 16 + g.integers(0, 16, n)].astype(np.float64)
    z = np.sort(g.uniform(3, 12, (s["offsets"].size, per)), 1).reshape(-1, 1)
    scales = np.exp(g.normal(-2.0, 0.4, (n, 3)))
    gro = np.where(np.arange(3) == g.integers(0, 4, n)[:, None], g.uniform(0.1, 0.95, (n, 1)), 1.0)
    a = gro * g.choice([-1.0, 1.0], (n, 3)) * scales  # R^T (o - mu), up to its length
    a /= np.linalg.norm(a, axis=1, keepdims=True)
    arc = np.concatenate([1 + (a * v).sum(1, keepdims=True), np.cross(a, v)], 1)  # the rotation that takes a to v
    arc /= np.linalg.norm(arc, axis=1, keepdims=True)
    half = g.uniform(0, np.pi, (n, 1))
    quats = _quat_mul(np.concatenate([np.cos(half), np.sin(half) * v], 1), arc)
    f32 = lambda x: np.ascontiguousarray(x, np.float32)
    s.update(means=f32(s["ro"][0, 0] - v * z), quats=f32(quats), scales=f32(scales), colors=f32(g.normal(0, 1, (n, 3))),
             opac=f32(g.uniform(0.006, 0.02, n)), flat=np.arange(n, dtype=np.int32),
             offsets=(np.arange(s["offsets"].size, dtype=np.int32) * per).reshape(s["offsets"].shape))
    out, work, T = _forward(s)
    grads = _image_grads(W, H, 3)
    ref = _oracle_bwd(s, np_(out[2]), np_(out[3]), grads)
    for kw in (dict(ray_grads=True), dict(ray_grads=False, pixels_per_lane=2), dict(ray_grads=False, pixels_per_lane=4)):
        got = _backward(s, out, work, T, grads, **kw)
        for name in ("v_means", "v_quats", "v_scales"):
            size = np.linalg.norm(ref[name], axis=1)
            usual = size > np.quantile(size, 0.2)
            err = np.linalg.norm(got[name] - ref[name], axis=1)
            assert (err[usual] <= 1e-3 * size[usual]).all(), (name, int((err[usual] > 1e-3 * size[usual]).sum()), kw)


@pytest.mark.parametrize("distance", [0.0, 1e-38, 1e-25, 3e-20, 1e-19, 3e-19, 1e-15])
@pytest.mark.parametrize("scale", [0.1, 30.0])
def test_gaussians_at_the_camera(distance, scale):
    """A Gaussian that the camera sits in, down to distances whose squares float32 does not hold."""
    W, H = 33, 20
    s = _scene(W, H, (16, 16), n=6, seed=4)
    g = np.random.default_rng(1)
    s["ro"][...] = 0.0
    d = g.normal(0, 1, (6, 3))
    s["means"][:] = distance * d / np.linalg.norm(d, axis=1, keepdims=True)
    s["scales"][:] = scale * g.uniform(0.5, 2.0, (6, 3))
    out, work, T = _forward(s)
    _check_images(out, _oracle_fwd(s), np.ones((H, W), bool))
    v = _image_grads(W, H, 3)
    ref = _oracle_bwd(s, np_(out[2]), np_(out[3]), v)
    for kw in (dict(ray_grads=True), dict(ray_grads=False, pixels_per_lane=2), dict(ray_grads=False, pixels_per_lane=4)):
        got = _backward(s, out, work, T, v, **kw)
        for k in ("v_opacity", "v_colors", "v_means"):
            assert np.linalg.norm(got[k] - ref[k]) <= 1e-3 * np.linalg.norm(ref[k]) + 1e-12, (k, kw)
        assert all(np.isfinite(x).all() for x in got.values())


@pytest.mark.parametrize("dynamic", [False, True])
@pytest.mark.parametrize("tile,cdim", [((8, 8), 3), ((8, 8), 17), ((5, 7), 33), ((16, 8), 17), ((12, 10), 32), ((16, 8), 1),
                                       ((13, 9), 33), ((32, 32), 16), ((32, 32), 17), ((32, 20), 9)])
def test_small_and_large_workgroups(tile, cdim, dynamic):
    """Tiles of one and two strips (one wavefront in the backward), whose workgroups have LDS of their own size, and
    large tiles of many channels; lists that end inside, at and past a batch."""
    W, H = 70, 45
    v = _image_grads(W, H, cdim)
    for n in (64, 130):
        s = _scene(W, H, tile, n=n, cdim=cdim, dynamic=dynamic, seed=n)
        out, work, T = _forward(s)
        _check_images(out, _oracle_fwd(s), np.ones((H, W), bool))
        ref = _oracle_bwd(s, np_(out[2]), np_(out[3]), v)
        for ray_grads in ((True, False) if cdim <= 16 else (True,)):
            _check_grads(_backward(s, out, work, T, v, ray_grads=ray_grads), ref)


@pytest.mark.parametrize("moving,dynamic", [(False, False), (True, False), (False, True)])
@pytest.mark.parametrize("what,value", [("opac", np.nan), ("opac", np.inf), ("means", np.nan), ("means", np.inf),
                                        ("quats", 0.0), ("quats", np.nan), ("scales", 0.0), ("scales", np.nan),
                                        ("scales", np.inf)])
def test_gaussians_that_are_no_numbers(what, value, moving, dynamic):
    """They reach the alpha test as they are: an alpha that is no number is 0.999, and a Gaussian of infinite extent
    has its opacity everywhere. (Depths are not compared: such a Gaussian's is no number.)"""
    W, H = 50, 37
    s = _scene(W, H, (16, 16), n=40, moving=moving, dynamic=dynamic)
    s["opac"] *= np.float32(0.3)
    s[what][17] = value
    out, work, T = _forward(s)
    _check_images(out, _oracle_fwd(s), np.ones((H, W), bool), depth=False)
