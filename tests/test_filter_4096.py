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
