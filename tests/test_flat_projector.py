"""The 2-D projector (fan and parallel beams) at the sizes where its layout
ends: one column and one pixel, wavefronts partly full, images of one row,
rays near the diagonal of the grid (where the walking axis changes from ray to
ray), and an image too large for the pair of layouts.

Tolerance: a ray's sum is a float chain of its segments, whose ends are float
parameters of up to the chord length; 2e-6 / 2e-5 is the bound that the cone
projector's tests derive for the same arithmetic."""
import numpy as np
import pytest

from conftest import errs, report

pytestmark = pytest.mark.gpu


# up to 6143 wavefronts of 64 rays a ray is split over four of them, and up to
# 128^2 pixels the image is read without its transpose
@pytest.mark.parametrize("nt,ns,bins,views", [(1, 1, 1, 4), (129, 130, 70, 7), (40, 33, 256, 1600), (1, 37, 63, 9), (41, 1, 64, 9), (40, 33, 65, 16),
                                              (64, 64, 130, 24), (257, 129, 200, 8)])
@pytest.mark.parametrize("beam", ["fan", "parallel"])
def test_flat_projector(ctx, oracle, nt, ns, bins, views, beam):
    import ctr
    size = (nt * 1.0, ns * 0.9)
    beta = 2 * np.pi / views * np.arange(1, views + 1) + 0.003   # 45-degree views nearly on the diagonal
    half = 0.62 * np.hypot(*size)
    pos = np.linspace(-half, half, bins) if bins > 1 else np.array([0.11])
    img = np.random.default_rng(nt + bins).random(nt * ns).astype(np.float32)
    print(f"[case] flat projector {beam} {nt}x{ns} {views}x{bins}", flush=True)
    if beam == "fan":
        a = (nt, ns, size, 1.3 * np.hypot(*size), beta, pos)
        got, ref = ctx.fan_fp(ctr.FanGeom(*a), img), oracle.fan_fp_exact(oracle.Fan(*a), img)
    else:
        a = (nt, ns, size, beta, pos)
        got, ref = ctx.par_fp(ctr.ParGeom(*a), img), oracle.par_fp_exact(oracle.Par(*a), img)
    e, m = errs(got, ref)
    report(f"flat_fp[{beam},{nt}x{ns}]", rel_l2=e, max_rel=m)
    assert e < 2e-6 and m < 2e-5


def test_flat_projector_infinite_pixel(ctx):
    """Rays away from an infinite pixel keep their values bit for bit."""
    import ctr
    beta = 2 * np.pi / 20 * np.arange(1, 21) + 0.01
    g = ctr.FanGeom(48, 40, (48.0, 40.0), 80.0, beta, 0.7 * (np.arange(110) - 54.5))
    img = np.random.default_rng(2).random(g.nvox).astype(np.float32)
    a = ctx.fan_fp(g, img)
    i, j = 17, 22
    img[j * 48 + i] = np.inf
    b = ctx.fan_fp(g, img)
    near = np.zeros((40, 48), np.float32)
    near[j - 1:j + 2, i - 1:i + 2] = 1.0     # a ray outside these nine pixels does not touch the pixel
    away = ctx.fan_fp(g, near.ravel()) == 0
    assert away.any() and np.array_equal(a[away], b[away])
    one = np.zeros(g.nvox, np.float32)
    one[j * 48 + i] = 1.0
    hit = ctx.fan_fp(g, one) > 1e-3
    assert hit.any() and not np.isfinite(b[hit]).any()


def test_projector_of_an_image_beyond_the_pair(ctx):
    """2^28 pixels and more take the cone kernel: the projection of ones is the chord."""
    import ctr
    import torch
    n = 16400
    g = ctr.ParGeom(n, n, (4.0, 4.0), np.array([0.0, 0.4, 0.9]), np.array([-1.0, -0.2, 0.0, 0.7]))
    got = ctx.par_fp(g, torch.ones(n * n, device="cuda")).cpu().numpy().reshape(3, 4)
    for a, th in enumerate(g.theta):
        for b, t in enumerate(g.t):
            c, s = np.cos(th), np.sin(th)
            lo, hi = -np.inf, np.inf
            for o, d in ((t * c, -s), (t * s, c)):
                if abs(d) > 1e-12:
                    u, v = sorted(((-2 - o) / d, (2 - o) / d))
                    lo, hi = max(lo, u), min(hi, v)
            # 33000 segments telescope to the chord: their rounding, 2^-24 of up to 5 mm each
            assert abs(got[a, b] - (hi - lo)) < 1e-3


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("views,bins", [(20, 110), (400, 1100)])
def test_flat_projector_of_a_pixel_that_is_not_finite(ctx, bad, views, bins):
    """It reaches the rays that cross it, and those alone: the others have the bits
    of the projection with a 0 in its place.  Few rays (split over wavefronts, the
    image as it is) and many; both beams."""
    import ctr
    ang = 2 * np.pi / views * np.arange(1, views + 1) + 0.01
    pos = 77.0 / bins * (np.arange(bins) - (bins - 1) / 2)
    for n in ((48, 40), (150, 141)):
        size = (48.0, 40.0)
        for name, g, run in (("fan", ctr.FanGeom(*n, size, 80.0, ang, pos), ctx.fan_fp),
                             ("parallel", ctr.ParGeom(*n, size, ang, pos), ctx.par_fp)):
            img = np.random.default_rng(2).random(g.nvox).astype(np.float32)
            for at in (0, 17 * n[0] + 22, n[0] * n[1] - 1):
                print(f"[case] {name} {n} {views} x {bins}, {bad} at {at}", flush=True)
                one = np.zeros(g.nvox, np.float32)
                one[at] = 1.0
                meets = run(g, one)
                keep, img[at] = img[at], 0.0
                clean = run(g, img)
                img[at] = bad
                got = run(g, img)
                img[at] = keep
                assert np.array_equal(got[meets == 0], clean[meets == 0])
                hit = meets > 1e-3 * size[0] / n[0]
                assert hit.any() and np.array_equal(got[hit], np.full(hit.sum(), bad, np.float32), equal_nan=True)
