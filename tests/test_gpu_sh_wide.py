"""The [3, K, N] colour kernels that take several Gaussians per thread, against the one-per-thread kernels.

The wide kernels run from degree 3 (the forward's without a mask) on large arrays whose length is a multiple of
their vector; one Gaussian more (an odd length) takes the kernels that the other tests hold against the oracle,
on the same values. Sizes: just above the backward's rule (48 MB of coefficients) with a last workgroup partly
filled and lengths of 2 modulo 4, and just above the forward's (192 MB). Lower degrees and masked forwards of
these sizes take the one-per-thread kernels either way.

Bound: every value is a sum of at most 25 products per channel, taken in the same order; contraction may
differ, so 2 x 25 x 2^-24 = 3e-6 of the sum of the terms' magnitudes, which is below 32 here; the position
gradient adds the basis derivatives' factors (below 64) over distances of at least 0.5. The origin's gradient
is a sum of all rows in another grouping: 1e-5 of the rows' summed magnitudes.
"""
import numpy as np
import pytest
import torch

from xsimgs_amd import _C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("degree,dc,masked,mega", [
    (3, False, True, 48), (3, True, False, 48), (1, False, False, 48), (4, True, True, 48), (0, False, True, 48),
    (3, False, False, 192), (3, True, True, 192), (4, False, True, 192), (2, False, True, 192),
    (3, True, False, 192), (4, False, False, 192), (4, True, False, 192), (4, False, False, 48),
])
def test_wide_matches_single(degree, dc, masked, mega):
    bands = (degree + 1) ** 2 - (1 if dc else 0)
    n = ((mega << 20) // (12 * bands) // 4 + 67) * 4 + (2 if mega == 48 or degree == 4 else 0)
    g = torch.Generator(device="cuda").manual_seed(degree * 10 + mega)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    pos = rnd(n + 1, 3)
    pos = pos / pos.norm(dim=1, keepdim=True) * (0.5 + 4 * torch.rand(n + 1, 1, generator=g, device="cuda"))
    origin = torch.tensor([0.01, -0.02, 0.03], device="cuda")
    coeffs, d_out = rnd(3, bands, n + 1), rnd(n + 1, 3)
    d_out[torch.rand(n + 1, generator=g, device="cuda") < 0.4] = 0.0
    base = rnd(3, n + 1) if dc else None
    words = (n + 1 + 31) // 32
    mask = torch.randint(-2 ** 31, 2 ** 31 - 1, (words,), generator=g, device="cuda", dtype=torch.int32) if masked else None
    if masked:
        mask[: words // 3] = 0
    cut = lambda t, d: None if t is None else t.narrow(d, 0, n).contiguous()
    one = _C.spherical_harmonics_fused_fwd(degree, origin, pos, coeffs, mask, True, base)
    wide = _C.spherical_harmonics_fused_fwd(degree, origin, cut(pos, 0), cut(coeffs, 2), mask, True, cut(base, 1))
    if masked:  # masked rows of the output are not written
        bits = np.unpackbits(mask.cpu().numpy().view(np.uint8), bitorder="little")[:n]
        keep = torch.from_numpy(bits != 0).cuda()
        one, wide = one[:n][keep], wide[keep]
    else:
        one = one[:n]
    assert float((one - wide).abs().max()) <= 3e-6 * 32
    a = _C.spherical_harmonics_fused_bwd(degree, origin, pos, coeffs, mask, True, d_out, base)
    b = _C.spherical_harmonics_fused_bwd(degree, origin, cut(pos, 0), cut(coeffs, 2), mask, True, cut(d_out, 0), cut(base, 1))
    for x, y, axis in ((a[0], b[0], 2), (a[1], b[1], 1), (a[2], b[2], 0)):
        if x is None or x.numel() == 0:
            continue
        x = x.narrow(axis, 0, n)
        assert float((x - y).abs().max()) <= 3e-6 * 64 * 2, axis
        assert torch.equal(x == 0, y == 0)
    rest = a[2][n].double()
    want = a[3].double().view(-1) + rest  # (the origin's gradient is minus the positions')
    assert float((b[3].double().view(-1) - want).abs().max()) <= 1e-5 * float(b[2].abs().sum())
