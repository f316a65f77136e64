"""The 2-D FBP backprojections where their layout ends: fewer views than
wavefronts, tiles partly outside the image, a detector that part of a tile
misses, bins too fine for the shadow of a tile to be held in registers, and
pixels seen from the source at more than 27 degrees.

Tolerances: 2e-5 / 2e-4 is the bound of the suite's FBP tests (a detector
coordinate of up to 101 bins carries a few float ulps, 1e-5 bins, and
the data change by up to 1 a bin).  Near the source w = D - s loses a factor
D / w <= 20 to cancellation and a bin coordinate 4 eps 20 x 42 bins/rad =
2e-4 bins: 1e-4 / 1e-3 there."""
import numpy as np
import pytest

from conftest import errs, report

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt,ns,views,bins,cover", [(1, 1, 2, 2, 1.0), (17, 3, 7, 40, 1.3), (16, 16, 8, 37, 0.45),
                                                    (33, 40, 9, 61, 0.45), (17, 3, 17, 90, 1.3)])
@pytest.mark.parametrize("descending", [False, True])
def test_par_fbp_tiles(ctx, oracle, nt, ns, views, bins, cover, descending):
    import ctr
    size = (nt * 1.0, ns * 0.9)
    theta = (np.pi / views * np.arange(views) + 0.01).astype(np.float32).astype(np.float64)
    t = (np.linspace(-0.5, 0.5, bins) * cover * np.hypot(*size) + 0.013).astype(np.float32).astype(np.float64)
    a = (nt, ns, size, theta, t[::-1].copy() if descending else t)
    g, og = ctr.ParGeom(*a), oracle.Par(*a)
    y = np.random.default_rng(nt + bins).random(g.nray).astype(np.float32)
    print(f"[case] parallel FBP {nt}x{ns} {views}x{bins}", flush=True)
    img = ctx.par_fbp(g, y)
    with oracle.interp_mode(1):
        ref = oracle.par_fbp_bp(og, oracle.par_filter(og, y).astype(np.float32))
    e, m = errs(img, ref)
    report(f"par_fbp[{nt}x{ns},{views}x{bins},desc={descending}]", rel_l2=e, max_rel=m)
    assert e < 2e-5 and m < 2e-4
    np.testing.assert_array_equal(ctx.par_fbp(g, y, out=img.copy(), flags=ctr.ACCUMULATE), img + img)


@pytest.mark.parametrize("nt,ns,views,distance,tol", [(1, 1, 2, 8.0, 2e-5), (9, 15, 7, 4.0, 2e-5), (40, 33, 19, 3.0, 2e-5),
                                                      (24, 24, 9, 1.05, 1e-4)])
@pytest.mark.parametrize("equiangular", [False, True])
def test_fan_fbp_tiles(ctx, oracle, nt, ns, views, distance, tol, equiangular):
    import ctr
    size = (nt * 1.0, ns * 0.9)
    half = 0.5 * np.hypot(*size)
    D = distance * half
    beta = (2 * np.pi / views * np.arange(views) + 0.01).astype(np.float32).astype(np.float64)
    if equiangular:
        p = D * np.tan(np.linspace(-1.2, 1.2, 101) if distance < 2 else np.linspace(-1, 1, 101) * 1.1 / distance)
    else:
        p = (np.linspace(-1.3, 1.3, 101) * (3.0 if distance < 2 else 1.0) * half).astype(np.float32).astype(np.float64)
    a = (nt, ns, size, D, beta, p)
    g, og = ctr.FanGeom(*a), oracle.Fan(*a)
    y = np.random.default_rng(nt + views).random(g.nray).astype(np.float32)
    print(f"[case] fan FBP {nt}x{ns} {views} views, D = {distance} half diagonals", flush=True)
    img = ctx.fan_fbp(g, y, detector=ctr.FAN_EQUIANGULAR if equiangular else ctr.FAN_FLAT)
    with oracle.interp_mode(1):
        ref = oracle.fan_fbp_bp(og, oracle.fan_filter(og, y, equiangular=equiangular).astype(np.float32),
                                equiangular=equiangular)
    e, m = errs(img, ref)
    report(f"fan_fbp[{nt}x{ns},D={distance},eq={equiangular}]", rel_l2=e, max_rel=m)
    assert e < tol and m < 10 * tol
