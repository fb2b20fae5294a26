"""The compositor's launch variants and batch remainders against the float64 oracle.

The forward takes two pixels per lane on grids of at least 8192 such wavefronts, one on others, and four
Gaussians per step on grids of at most 4096 wavefronts; the backward four or two pixels per lane, with its
batches of one Gaussian per thread or (many channels) of 64. Every tile lists the same Gaussians in depth
order, so the list lengths put the end of a list at, before and after the batches' and steps' ends; the
image sizes leave tiles one pixel wide, whose rays give no direction of their own.

Bounds. Renders: 1e-4 absolute, the suite's bar, on all but one pixel in ten thousand: a float32 alpha (error
about 1e-6) or transmittance falls on the other side of its threshold in fewer. Gradients: 1e-3 of an array's
norm, the suite's relative bar (the oracle is given the same float32 alpha image, whose 6e-8 a nearly opaque
pixel's remaining transmittance of 1e-4 turns into 6e-4).
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from xsimgs_amd import _C
from tests._util import np_

pytestmark = pytest.mark.gpu


def _scene(W, H, tile, n, cdim, shutter=False, seed=0):
    g = np.random.default_rng(seed)
    listed, n = n, max(n, 1)  # (length 0: a Gaussian that no tile lists)
    z = np.sort(g.uniform(3.0, 30.0, n))
    f = 0.9 * W
    means = np.stack([g.uniform(-0.55, 0.55, n) * z, g.uniform(-0.55, 0.55, n) * H / W * z, z], -1)
    scales = np.exp(g.normal(np.log(0.12), 0.5, (n, 3))) * z[:, None] / 10
    quats = g.normal(0, 1, (n, 4))
    opac = g.uniform(0.02, 0.9995, n)
    colors = g.normal(0, 1, (n, cdim))
    x = (np.arange(W) + 0.5 - W / 2) / f
    y = (np.arange(H) + 0.5 - H / 2) / f
    rd = np.stack([np.broadcast_to(x, (H, W)), np.broadcast_to(y[:, None], (H, W)), np.ones((H, W))], -1)
    rd /= np.linalg.norm(rd, axis=-1, keepdims=True)
    ro = np.zeros((H, W, 3)) + [0.1, -0.2, 0.05]
    if shutter:  # a camera that moves from row to row
        ro = ro + (np.arange(H) / H)[:, None, None] * np.array([0.05, 0.0, -0.02])
    ntx, nty = -(-W // tile[0]), -(-H // tile[1])
    flat = np.tile(np.arange(listed, dtype=np.int32), ntx * nty)
    offsets = (np.arange(ntx * nty, dtype=np.int32) * listed).reshape(nty, ntx)
    c = lambda a: np.ascontiguousarray(a, np.float32)
    return [c(a) for a in (means, quats, scales, colors, opac, ro, rd)] + [offsets, flat]


def _run(s, W, H, tile):
    means, quats, scales, colors, opac, ro, rd, offsets, flat = [torch.from_numpy(a).cuda() for a in s]
    work = torch.empty(offsets.numel(), dtype=torch.int32, device="cuda")
    out = _C.rasterize_eval3d_fwd(means, quats, scales, colors.unsqueeze(0), opac.view(1, -1), W, H, *tile, ro, rd,
                                  offsets, flat, tile_work=work)
    return out, work


SIZES = [  # image, tile: two pixels per lane; one; one and four Gaussians per step; one strip per tile
    ((1009, 1025), (16, 16), [130]),
    ((700, 600), (16, 16), [129, 257]),
    ((97, 81), (16, 16), [0, 1, 3, 4, 5, 63, 64, 65, 255, 256, 257]),
    ((1000, 900), (8, 8), [65]),
    ((65, 50), (32, 32), [511, 513]),
]


@pytest.mark.parametrize("shutter", [False, True])
@pytest.mark.parametrize("size,tile,lengths", SIZES)
def test_forward_variants(size, tile, lengths, shutter):
    W, H = size
    for n in lengths:
        s = _scene(W, H, tile, n, 3, shutter, seed=n)
        (rgb, depth, alpha, last), work = _run(s, W, H, tile)
        ref = O.eval3d_fwd(*s[:7], s[7], s[8], *tile, prec="f64")
        for got, want in zip((rgb, depth, alpha), ref[:3]):
            bad = np.abs(np_(got) - want) > 1e-4 * np.maximum(1.0, np.abs(want))
            assert bad.mean() <= 1e-4, (n, bad.mean())
        assert (np_(last) != ref[3]).mean() <= 1e-4, n
        # the tile's work: its list up to the largest last id of its pixels
        nty, ntx = s[7].shape
        pad = np.zeros((nty * tile[1], ntx * tile[0]), np.int64)
        pad[:H, :W] = np_(last)
        top = pad.reshape(nty, tile[1], ntx, tile[0]).max(axis=(1, 3)).reshape(-1)
        first = s[7].reshape(-1)
        assert np.array_equal(np_(work), np.maximum(0, np.minimum(first + n - 1, top) - first + 1))


GRADS = [  # image, tile, channels, list length
    ((97, 81), (16, 16), 3, 0), ((97, 81), (16, 16), 3, 1), ((97, 81), (16, 16), 3, 64), ((97, 81), (16, 16), 3, 129),
    ((97, 81), (16, 16), 32, 65), ((97, 81), (16, 16), 33, 64), ((97, 81), (8, 8), 17, 63), ((65, 50), (32, 32), 16, 257),
    ((65, 50), (32, 32), 32, 70),
]


@pytest.mark.parametrize("shutter", [False, True])
@pytest.mark.parametrize("size,tile,cdim,n", GRADS)
def test_backward_variants(size, tile, cdim, n, shutter):
    W, H = size
    s = _scene(W, H, tile, n, cdim, shutter, seed=100 + n)
    (_, _, alpha, last), work = _run(s, W, H, tile)
    g = np.random.default_rng(7)
    v = [g.normal(0, 1e-3, shape).astype(np.float32) for shape in ((H, W, cdim), (H, W), (H, W))]
    means, quats, scales, colors, opac, ro, rd, offsets, flat = s
    ref = O.eval3d_bwd(means, quats, scales, colors, opac, ro, rd, offsets, flat, np_(alpha), np_(last), *v, *tile,
                       prec="f64")
    T = [torch.from_numpy(a).cuda() for a in s]
    V = [torch.from_numpy(a).cuda() for a in v]
    for ray_grads in ((True, False) if cdim <= 16 else (True,)):
        for ppl in ((0,) if ray_grads else (2, 4)):
            got = _C.rasterize_eval3d_bwd(T[0], T[2], T[1], T[4], T[3], T[5], T[6], *tile, T[7], T[8], alpha, last, *V,
                                          ray_grads=ray_grads, pixels_per_lane=ppl, tile_work=work)
            names = ["v_means", "v_quats", "v_scales", "v_opacity", "v_colors"] + (["v_ray_o", "v_ray_d"] if ray_grads else [])
            for name, x in zip(names, got):
                want = ref[name]
                err = np.linalg.norm(np_(x).reshape(-1) - want.reshape(-1))
                assert err <= 1e-3 * np.linalg.norm(want) + 1e-12, (name, ray_grads, ppl, err, np.linalg.norm(want))
