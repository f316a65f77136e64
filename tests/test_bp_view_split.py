"""Backprojection and exact adjoint of small volumes with the views split over
sets of blocks: too few views for a split, shares with a remainder, one tile
and several ragged ones.  Bounds: the ones of the suite's single-pass FDK,
reference backprojection and adjoint (the split changes the order of the sums
only)."""
import numpy as np
import pytest

from conftest import errs, report

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("views", [2, 7, 8, 9, 41])
@pytest.mark.parametrize("shape", [(16, 16, 16), (21, 17, 19)])
def test_split_views(ctx, oracle, shape, views):
    import ctr
    nt, ns, nz = shape
    beta = (2 * np.pi / views * np.arange(views) + 0.1).astype(np.float32)
    p, xi = (np.linspace(-1, 1, n).astype(np.float32) * np.float32(16.0) for n in (37, 33))
    a = (nt, ns, nz, (nt * 1.0, ns * 1.1, nz * 0.9), 60.0, beta, p, xi)
    g, og = ctr.ConeGeom(*a), oracle.Cone(*a)
    y = np.random.default_rng(views).standard_normal(g.nray).astype(np.float32)
    print(f"[case] split backprojection {shape}, {views} views", flush=True)
    img = ctx.fdk_bp(g, y)
    with oracle.interp_mode(1):
        e, m = errs(img, oracle.fdk_bp(og, y))
        e2, m2 = errs(ctx.cone_bp_ref(g, y), oracle.cone_bp_ref(og, y))
    report(f"split_bp[{shape},{views}]", rel_l2=e, max_rel=m, ref_rel_l2=e2, ref_max_rel=m2)
    assert e < 3e-5 and m < 1e-4 and e2 < 3e-5 and m2 < 1e-4
    np.testing.assert_array_equal(ctx.fdk_bp(g, y, out=img.copy(), flags=ctr.ACCUMULATE), img + img)


@pytest.mark.parametrize("views", [2, 7, 8, 9, 41])
@pytest.mark.parametrize("shape", [(16, 16, 4), (21, 17, 19)])
def test_split_adjoint(ctx, oracle, shape, views):
    import ctr
    nt, ns, nz = shape
    beta = (2 * np.pi / views * np.arange(views) + 0.1).astype(np.float32)
    p, xi = (np.linspace(-1, 1, n).astype(np.float32) * np.float32(16.0) for n in (37, 33))
    a = (nt, ns, nz, (nt * 1.0, ns * 1.1, nz * 0.9), 60.0, beta, p, xi)
    g, og = ctr.ConeGeom(*a), oracle.Cone(*a)
    y = np.random.default_rng(views).random(g.nray).astype(np.float32)
    print(f"[case] split adjoint {shape}, {views} views", flush=True)
    vol = ctx.cone_bp_adjoint(g, y)
    e, m = errs(vol, oracle.cone_adjoint(og, y))
    report(f"split_adjoint[{shape},{views}]", rel_l2=e, max_rel=m)
    assert e < 1e-4 and m < 1e-3
    np.testing.assert_array_equal(ctx.cone_bp_adjoint(g, y, out=vol.copy(), flags=ctr.ACCUMULATE), vol + vol)


@pytest.mark.parametrize("pitch", [0.01, 1e-9])
@pytest.mark.parametrize("nz", [4, 6])
def test_adjoint_of_slices_far_off_the_rows(ctx, oracle, nz, pitch):
    """Few fine rows and thick slices: the slices of a tile that the rows miss lie
    hundreds of rows (and more than an int counts) away from the staged ones.
    Rows of 1e-9 mm are finer than a float knows a face of a 6 mm slice (4e-7 mm),
    so that only the slices which no ray comes near have a value to hold to."""
    import ctr
    beta = (2 * np.pi / 9 * np.arange(9) + 0.1).astype(np.float32)
    p = (0.8 * (np.arange(37) - 18)).astype(np.float32)
    xi = (pitch * (np.arange(20) - 9.3)).astype(np.float32)
    a = (16, 17, nz, (16.0, 17.0, 6.0 * nz), 60.0, beta, p, xi)
    g, og = ctr.ConeGeom(*a), oracle.Cone(*a)
    y = np.random.default_rng(nz).random(g.nray).astype(np.float32)
    print(f"[case] adjoint of {nz} slices of 6 mm, 20 rows of {pitch} mm", flush=True)
    vol, ref = ctx.cone_bp_adjoint(g, y), oracle.cone_adjoint(og, y)
    if pitch < 1e-6:
        slices = np.asarray(vol).reshape(g.vol_shape).any(axis=(1, 2))
        assert np.isfinite(vol).all() and list(np.flatnonzero(slices)) == [nz // 2 - 1, nz // 2]
        return
    e, m = errs(vol, ref)
    report(f"thick_slices[{nz},{pitch}]", rel_l2=e, max_rel=m)
    assert e < 1e-4 and m < 1e-3


@pytest.mark.parametrize("rows,columns", [(400, 40), (40, 400)])
def test_backprojection_of_tall_and_wide_footprints(ctx, oracle, rows, columns):
    """Footprints larger than LDS holds: all views in one set, from memory."""
    import ctr
    beta = (2 * np.pi / 40 * np.arange(40) + 0.1).astype(np.float32)
    p, xi = (np.linspace(-1, 1, n).astype(np.float32) * np.float32(26.0) for n in (columns, rows))
    a = (24, 21, 33, (24.0, 23.1, 29.7), 60.0, beta, p, xi)
    g, og = ctr.ConeGeom(*a), oracle.Cone(*a)
    y = np.random.default_rng(rows).random(g.nray).astype(np.float32)
    print(f"[case] backprojection, 40 views of {rows} x {columns}", flush=True)
    img = ctx.fdk_bp(g, y)
    with oracle.interp_mode(1):
        e, m = errs(img, oracle.fdk_bp(og, y))
        e2, m2 = errs(ctx.cone_bp_ref(g, y), oracle.cone_bp_ref(og, y))
    report(f"bp_beyond_lds[{rows}x{columns}]", rel_l2=e, max_rel=m, ref_rel_l2=e2, ref_max_rel=m2)
    assert e < 3e-5 and m < 1e-4 and e2 < 3e-5 and m2 < 1e-4
    np.testing.assert_array_equal(ctx.fdk_bp(g, y, out=img.copy(), flags=ctr.ACCUMULATE), img + img)
