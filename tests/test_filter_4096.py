"""The flat-detector row filters by a transform of 4096 (1025 to 2048 bins): the
shortest and longest rows, an odd number of rows, and every mode, against the
FP64 oracle.  Bound: the suite's for row filters (FP64 sums rounded to float)."""
import numpy as np
import pytest

from conftest import errs, report

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bins", [1024, 1025, 1280, 2047, 2048])
@pytest.mark.parametrize("filt", [0, 1])
def test_long_rows(ctx, oracle, bins, filt):
    import ctr
    rng = np.random.default_rng(bins)
    t = (0.05 * (np.arange(bins) - 0.5 * (bins - 1))).astype(np.float32).astype(np.float64)
    beta = np.deg2rad(np.arange(1, 6) * 72.0).astype(np.float32)
    b64 = beta.astype(np.float64)
    print(f"[case] filter of {bins} bins", flush=True)
    got = {}
    a = (8, 8, (8.0, 8.0), b64, t)
    g, og = ctr.ParGeom(*a), oracle.Par(*a)
    y = rng.random(g.nray).astype(np.float32)
    got["parallel"] = ctx.par_filter(g, y, filt=filt), oracle.par_filter(og, y, filt=filt)
    a = (8, 8, (8.0, 8.0), 1000.0, b64, t)
    got["fan"] = ctx.fan_filter(ctr.FanGeom(*a), y, filt=filt), oracle.fan_filter(oracle.Fan(*a), y, filt=filt)
    a = (8, 8, 4, (8.0, 8.0, 4.0), 1000.0, beta, t.astype(np.float32), np.array([-0.5, 0.0, 0.5], np.float32))
    y = rng.random(5 * 3 * bins).astype(np.float32)
    got["cone"] = ctx.cone_filter(ctr.ConeGeom(*a), y, filt=filt), oracle.cone_filter(oracle.Cone(*a), y, filt=filt)
    for name, (x, ref) in got.items():
        e, m = errs(x, ref)
        report(f"filter[{name},{bins},f={filt}]", rel_l2=e, max_rel=m)
        assert e < 1e-6 and m < 1e-5


@pytest.mark.parametrize("bins", [1025, 1500, 2048])
def test_a_row_keeps_its_infinities_to_itself(ctx, oracle, bins):
    """Rows with a NaN or an infinity are filtered by the direct sums: NaN and
    infinite where those are, and the other rows as if the bad ones were zero,
    bit for bit; also in place."""
    import ctr
    import torch
    rng = np.random.default_rng(bins)
    t = (0.05 * (np.arange(bins) - 0.5 * (bins - 1))).astype(np.float32).astype(np.float64)
    beta = np.deg2rad(np.arange(1, 8) * 50.0)
    xi = np.array([-0.5, 0.5], np.float32)
    forms = {
        "parallel": (ctr.ParGeom, oracle.Par, (8, 8, (8.0, 8.0), beta, t), ctx.par_filter, oracle.par_filter),
        "fan": (ctr.FanGeom, oracle.Fan, (8, 8, (8.0, 8.0), 1000.0, beta, t), ctx.fan_filter, oracle.fan_filter),
        "cone": (ctr.ConeGeom, oracle.Cone, (8, 8, 4, (8.0, 8.0, 4.0), 1000.0, beta[:4].astype(np.float32),
                                             t.astype(np.float32), xi), ctx.cone_filter, oracle.cone_filter),
    }
    clean8 = rng.random((8, bins)).astype(np.float32)
    clean8[[1, 2, 6]] = 0.0
    y = y8 = clean8.copy()
    y[[1, 2, 6]] = rng.random((3, bins)).astype(np.float32)
    y[1, bins - 1], y[2, 700], y[6, 0], y[6, 9] = np.nan, -np.inf, np.inf, np.inf   # partners 0, 3 and 7 or none
    for name, (G, O, a, run, ref) in forms.items():
        print(f"[case] {name} {bins}", flush=True)
        g = G(*a)
        rows = g.nray // bins
        clean, y, good = clean8[:rows], y8[:rows], [0, 3, 4, 5, 7][:rows - 3]
        want = np.asarray(ref(O(*a), y.ravel())).reshape(rows, bins)
        base = np.asarray(run(g, clean.ravel())).reshape(rows, bins)
        x = torch.from_numpy(y.ravel()).cuda()
        run(g, x, out=x)
        for got in (np.asarray(run(g, y.ravel())), x.cpu().numpy()):
            got = got.reshape(rows, bins)
            assert np.array_equal(got[good], base[good]), name
            for i in (1, 2, 6):
                assert np.array_equal(np.isnan(got[i]), np.isnan(want[i])), (name, i)
                assert np.array_equal(got[i][~np.isnan(got[i])], want[i][~np.isnan(want[i])].astype(np.float32)), (name, i)


@pytest.mark.parametrize("bins", [1025, 1500, 2048])
@pytest.mark.parametrize("filt", [0, 1])
def test_a_row_keeps_its_rounding_to_itself(ctx, oracle, bins, filt):
    """Rows of every size from 1e-30 to 1e30 and rows of zeros side by side: each is
    held to the suite's bound by its own size, and zeros come out as zeros."""
    import ctr
    rng = np.random.default_rng(bins)
    t = (0.05 * (np.arange(bins) - 0.5 * (bins - 1))).astype(np.float32).astype(np.float64)
    beta = np.deg2rad(np.arange(1, 10) * 40.0)
    sizes = np.array([1.0, 1e30, 1e-30, 0.0, 0.0, 3e4, 1e12, 1.0, 1e-20], np.float32)
    y = sizes[:, None] * rng.random((9, bins)).astype(np.float32)
    y[7, bins // 3:] = 0.0
    three = (8, 8, 4, (8.0, 8.0, 4.0), 1000.0, beta[:3].astype(np.float32), t.astype(np.float32),
             np.array([-0.5, 0.0, 0.5], np.float32))
    forms = {
        "parallel": (ctr.ParGeom, oracle.Par, (8, 8, (8.0, 8.0), beta, t), ctx.par_filter, oracle.par_filter),
        "fan": (ctr.FanGeom, oracle.Fan, (8, 8, (8.0, 8.0), 1000.0, beta, t), ctx.fan_filter, oracle.fan_filter),
        "cone": (ctr.ConeGeom, oracle.Cone, three, ctx.cone_filter, oracle.cone_filter),
    }
    for name, (G, O, a, run, ref) in forms.items():
        print(f"[case] {name} {bins} filter {filt}", flush=True)
        got = np.asarray(run(G(*a), y.ravel(), filt=filt)).reshape(9, bins)
        want = np.asarray(ref(O(*a), y.ravel(), filt=filt)).reshape(9, bins)
        for i, size in enumerate(sizes):
            if size == 0.0:
                assert not got[i].any() and not np.signbit(got[i]).any()
                continue
            e, m = errs(got[i].astype(np.float64) / size, want[i].astype(np.float64) / size)
            report(f"rows of {size}[{name},{bins},f={filt}]", rel_l2=e, max_rel=m)
            assert e < 1e-6 and m < 1e-5
