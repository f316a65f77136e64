"""The projector by detector columns (forced with CTR_FP_COLUMNS=1) at the
sizes where its paths end: row counts around a wavefront, single slices, lists
shorter than a block, rays that leave through the top and the bottom, cones so
steep that a block of cells holds several z crossings, rows closer and wider
than the 64-slice window, descending detectors, lines that miss the box.

Tolerance: the bound of the cone projector's tests (float crossing parameters,
one rounding each): rel-L2 2e-6, largest error 2e-5 of the largest integral."""
import numpy as np
import pytest

from conftest import errs, report

pytestmark = pytest.mark.gpu

CASES = {
    # name: nt, ns, nz, size, D, views, columns, column pitch, rows, row pitch
    "row": (20, 18, 12, (20.0, 18.0, 12.0), 60.0, 9, 33, 0.9, 1, 0.7),
    "rows63": (24, 20, 30, (24.0, 20.0, 30.0), 70.0, 7, 37, 0.8, 63, 0.5),
    "rows65": (24, 20, 30, (24.0, 20.0, 30.0), 70.0, 18, 70, 0.5, 65, 0.5),
    "rows130": (33, 40, 64, (33.0, 40.0, 64.0), 110.0, 17, 21, 1.7, 130, 0.55),
    "one_slice": (16, 16, 1, (16.0, 16.0, 2.0), 50.0, 5, 20, 0.9, 66, 0.05),
    "one_voxel": (1, 1, 1, (1.0, 1.0, 1.0), 5.0, 8, 9, 0.3, 12, 0.2),
    "out_of_top": (40, 40, 8, (40.0, 40.0, 4.0), 90.0, 12, 40, 1.2, 64, 0.4),
    "steep": (30, 30, 30, (30.0, 30.0, 30.0), 40.0, 11, 40, 1.0, 64, 1.0),
    "very_steep": (24, 24, 96, (24.0, 24.0, 24.0), 30.0, 11, 30, 1.0, 64, 1.2),
    "wide_rows": (24, 24, 200, (24.0, 24.0, 24.0), 300.0, 9, 30, 1.0, 80, 0.4),
    "misses": (16, 12, 10, (16.0, 12.0, 10.0), 60.0, 6, 80, 1.0, 20, 1.0),
    "descending": (20, 24, 16, (20.0, 24.0, 16.0), 70.0, 13, 40, -0.9, 40, -0.6),
    "thin": (200, 3, 20, (20.0, 6.0, 20.0), 50.0, 8, 50, 0.5, 30, 0.8),
}


def _geom(case, lib):
    nt, ns, nz, size, D, nb, np_, pp, nx, px = CASES[case]
    beta = (2 * np.pi / nb * np.arange(1, nb + 1)).astype(np.float32)
    p = (pp * (np.arange(np_) - (np_ - 1) / 2) + 0.03).astype(np.float32)
    xi = (px * (np.arange(nx) - (nx - 1) / 2) + 0.02).astype(np.float32)
    return lib(nt, ns, nz, size, D, beta, p, xi)


@pytest.fixture
def columns(monkeypatch):
    monkeypatch.setenv("CTR_FP_COLUMNS", "1")


@pytest.mark.parametrize("case", CASES)
def test_column_projector(ctx, oracle, columns, case):
    import ctr
    g, og = _geom(case, ctr.ConeGeom), _geom(case, oracle.Cone)
    vol = np.random.default_rng(len(case)).random(g.nvox).astype(np.float32)
    print(f"[case] columns {case} {g.vol_shape} {g.proj_shape}", flush=True)
    e, m = errs(ctx.cone_fp(g, vol), oracle.cone_fp_exact(og, vol))
    report(f"columns[{case}]", rel_l2=e, max_rel=m)
    assert e < 2e-6 and m < 2e-5


def test_column_projector_of_ones(ctx, oracle, columns):
    """Lengths telescope: the projection of ones is the chord to the rounding of its ends."""
    import ctr
    g, og = _geom("rows130", ctr.ConeGeom), _geom("rows130", oracle.Cone)
    e, m = errs(ctx.cone_fp(g, np.ones(g.nvox, np.float32)), oracle.cone_rowsum(og))
    assert e < 2e-7 and m < 1e-6


def test_columns_leave_sirt_alone(ctx, monkeypatch):
    """The residual pass of SIRT keeps the slab walk, whose rounding its residual
    history shows: iterates and history do not depend on the projector's kernel."""
    import ctr
    g = _geom("rows130", ctr.ConeGeom)
    vol = np.random.default_rng(4).random(g.nvox).astype(np.float32)
    monkeypatch.setenv("CTR_FP_COLUMNS", "0")
    b = ctx.cone_fp(g, vol)
    x0, r0, s0 = ctx.sirt3d(g, b, 2)
    monkeypatch.setenv("CTR_FP_COLUMNS", "1")
    x1, r1, s1 = ctx.sirt3d(g, b, 2)
    assert np.array_equal(x1, x0) and np.array_equal(r1, r0) and np.array_equal(s1, s0)


OFF_CENTRE = {
    # name: nt, ns, nz, size, D, rows, row pitch, rows the detector is shifted by.
    # All but the last two have a wavefront whose first and last row lie on both
    # sides of the source plane, one farther out than the other, more slices apart
    # than the shared window holds, or close to it, where the line leaves the
    # volume; "fits" has the same within the window.
    "one_chunk_up": (256, 256, 80, (256.0, 256.0, 80.0), 600.0, 64, 1.65, 18.5),
    "one_chunk_down": (256, 256, 80, (256.0, 256.0, 80.0), 600.0, 64, 1.65, -18.5),
    "fine_up": (256, 256, 80, (256.0, 256.0, 80.0), 600.0, 64, 1.3, 16.0),
    "fine_down": (256, 256, 80, (256.0, 256.0, 80.0), 600.0, 64, 1.3, -16.0),
    "near_the_source": (128, 128, 80, (128.0, 128.0, 80.0), 205.0, 128, 1.0, -16.0),
    "three_chunks": (256, 256, 80, (256.0, 256.0, 80.0), 600.0, 191, 1.1, 15.0),
    "centred": (256, 256, 100, (256.0, 256.0, 100.0), 600.0, 246, 2.5, 0.0),
    "descending": (256, 256, 80, (256.0, 256.0, 80.0), 600.0, 191, -1.1, 15.0),
    "fits": (256, 256, 80, (256.0, 256.0, 80.0), 600.0, 64, 0.55, 12.0),
    "one_side": (256, 256, 80, (256.0, 256.0, 80.0), 600.0, 64, 1.1, 32.5),
}


def _off_centre(case, lib, views, columns):
    nt, ns, nz, size, D, nx, px, shift = OFF_CENTRE[case]
    beta = (np.pi / 4 + 2 * np.pi / views * np.arange(views)).astype(np.float32)
    p = (150.0 / columns * (np.arange(columns) - (columns - 1) / 2) + 0.03).astype(np.float32)
    xi = (px * (np.arange(nx) - (nx - 1) / 2 + shift)).astype(np.float32)
    return lib(nt, ns, nz, size, D, beta, p, xi)


@pytest.mark.parametrize("case", OFF_CENTRE)
def test_rows_on_both_sides_of_the_source_plane(ctx, oracle, columns, case):
    import ctr
    g, og = _off_centre(case, ctr.ConeGeom, 3, 9), _off_centre(case, oracle.Cone, 3, 9)
    vol = np.random.default_rng(len(case)).random(g.nvox).astype(np.float32)
    print(f"[case] columns off centre {case} {g.vol_shape} {g.proj_shape}", flush=True)
    e, m = errs(ctx.cone_fp(g, vol), oracle.cone_fp_exact(og, vol))
    report(f"columns_off_centre[{case}]", rel_l2=e, max_rel=m)
    assert e < 2e-6 and m < 2e-5


@pytest.mark.parametrize("case", ["fine_up", "fine_down"])
def test_off_centre_rows_by_the_librarys_own_rule(ctx, oracle, case):
    """Enough wavefronts and slices for the library to take the columns by itself."""
    import ctr
    g, og = _off_centre(case, ctr.ConeGeom, 121, 101), _off_centre(case, oracle.Cone, 121, 101)
    vol = np.random.default_rng(7).random(g.nvox).astype(np.float32)
    print(f"[case] columns by rule {case} {g.vol_shape} {g.proj_shape}", flush=True)
    e, m = errs(ctx.cone_fp(g, vol), oracle.cone_fp_exact(og, vol))
    report(f"columns_by_rule[{case}]", rel_l2=e, max_rel=m)
    assert e < 2e-6 and m < 2e-5


@pytest.mark.parametrize("depth", [6e-7, 1e-44])
def test_rows_far_off_thin_slices(ctx, oracle, columns, depth):
    """Six slices whose thickness is next to nothing: the rows that miss them pass
    tens of millions of their planes, were these to go on, or planes so close that
    a float has no distance for them.  Rays end at the top and the bottom slice."""
    import ctr
    beta = (2 * np.pi / 5 * np.arange(5) + 0.1).astype(np.float32)
    p = (0.9 * (np.arange(30) - 14.5) + 0.03).astype(np.float32)
    inside = np.array([-1.15, -0.9, -0.4, 0.0, 0.3, 0.8, 1.2]) * 0.5 * depth
    xi = np.unique(np.concatenate([np.linspace(-15, -0.25, 30), inside, np.linspace(0.5, 15, 33)]).astype(np.float32))
    a = (24, 20, 6, (24.0, 20.0, depth), 70.0, beta, p, xi)
    g, og = ctr.ConeGeom(*a), oracle.Cone(*a)
    vol = np.random.default_rng(5).random(g.nvox).astype(np.float32)
    print(f"[case] columns, six slices in {depth} mm, {len(xi)} rows", flush=True)
    got, ref = ctx.cone_fp(g, vol), oracle.cone_fp_exact(og, vol)
    if depth < 1e-40:   # thinner than the oracle's own arithmetic: the rows off the volume only
        off = np.abs(np.broadcast_to(xi[None, :, None], g.proj_shape)) > 0.1
        assert not np.asarray(got).reshape(g.proj_shape)[off].any()
        return
    e, m = errs(got, ref)
    report(f"columns_thin[{depth}]", rel_l2=e, max_rel=m)
    assert e < 2e-6 and m < 2e-5


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("case", ["rows130", "rows65", "steep", "very_steep", "wide_rows"])
def test_a_voxel_that_is_not_finite(ctx, columns, case, bad):
    """It reaches the rays that cross it, and those alone: the others have the bits
    of the projection with a 0 in its place."""
    import ctr
    g = _geom(case, ctr.ConeGeom)
    nz, ns, nt = g.vol_shape
    vol = np.random.default_rng(3).random(g.vol_shape).astype(np.float32)
    crossed = 0
    for at in ((nz // 2, ns // 2, nt // 3), (nz - 1, ns // 2, nt // 2), (0, 0, 0)):
        print(f"[case] {case} {bad} at {at}", flush=True)
        one = np.zeros(g.vol_shape, np.float32)
        one[at] = 1.0
        meets = ctx.cone_fp(g, one.ravel())
        vol[at] = 0.0
        clean = ctx.cone_fp(g, vol.ravel())
        vol[at] = bad
        got = ctx.cone_fp(g, vol.ravel())
        vol[at] = 0.5
        assert np.array_equal(got[meets == 0], clean[meets == 0])
        hit = meets > 1e-4 * meets.max() if meets.any() else np.zeros(len(meets), bool)
        assert np.array_equal(got[hit], np.full(hit.sum(), bad, np.float32), equal_nan=True)
        crossed += hit.sum()
    assert crossed


@pytest.mark.parametrize("depth", [18.400000000000002, 31.2, 36.800000000000004, 80.0])
def test_level_rays_between_two_slices(ctx, oracle, columns, depth):
    """The middle one of an odd number of rows runs along the plane between the two
    middle slices: it takes the upper one, as in the slab walk and the matrix, also
    where depth / 2 times the reciprocal of the slice height rounds below it."""
    import ctr
    beta = (2 * np.pi / 5 * np.arange(5) + 0.1).astype(np.float32)
    p = (0.9 * (np.arange(30) - 14.5) + 0.03).astype(np.float32)
    xi = (0.31 * (np.arange(65) - 32)).astype(np.float32)
    a = (24, 20, 80, (24.0, 20.0, depth), 70.0, beta, p, xi)
    g, og = ctr.ConeGeom(*a), oracle.Cone(*a)
    vol = np.random.default_rng(6).random(g.nvox).astype(np.float32)
    print(f"[case] columns, level rays, 80 slices in {depth} mm", flush=True)
    e, m = errs(ctx.cone_fp(g, vol), oracle.cone_fp_exact(og, vol))
    report(f"columns_level[{depth}]", rel_l2=e, max_rel=m)
    assert e < 2e-6 and m < 2e-5
