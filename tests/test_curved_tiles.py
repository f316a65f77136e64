"""The curved-detector backprojection where its paths meet: tiles of every
depth with a ragged last one, one tile with its views split over sets of
blocks and many, footprints inside the detector and across its rows, of up to
96 and up to 128 channels, and cones thinner and wider than the weight's
series covers.  Bounds: the suite's for this backprojection."""
import numpy as np
import pytest

from conftest import errs, report

pytestmark = pytest.mark.gpu


#   voxels, slice height, source distance, channel pitch, row pitch, rows, views
@pytest.mark.parametrize("nt,ns,nz,rz,D,dg,dx,rows,views", [
    (16, 16, 4, 0.5, 400.0, 0.0008, 0.9, 24, 5),        # one tile, fewer views than a split
    (33, 17, 25, 0.5, 400.0, 0.0008, 0.9, 40, 41),      # thin cone, all rows on the detector
    (33, 17, 27, 0.5, 400.0, 0.0008, 0.9, 17, 41),      # rows off the detector
    (20, 16, 11, 0.5, 400.0, 0.00053, 0.9, 24, 23),     # footprints of 97 to 128 channels
    (20, 16, 33, 1.5, 150.0, 0.0021, 1.4, 96, 23),      # wide cone
    (20, 16, 9, 6.0, 400.0, 0.0008, 0.9, 120, 23),      # slices far apart: many rows a slice
])
def test_curved_tiles(ctx, oracle, nt, ns, nz, rz, D, dg, dx, rows, views):
    _compare(ctx, oracle, nt, ns, nz, rz, D, dg, dx, rows, views)


@pytest.mark.parametrize("nz,rows,D,dg", [
    (10, 40, 400.0, 0.0008), (12, 14, 400.0, 0.0008), (16, 40, 400.0, 0.0008), (20, 14, 400.0, 0.0008),
    (25, 40, 400.0, 0.0008), (25, 14, 400.0, 0.0008), (31, 40, 400.0, 0.0008), (32, 14, 400.0, 0.0008),
    (25, 40, 450.0, 0.00053),      # footprints of 97 to 128 channels
])
def test_deep_tiles(ctx, oracle, nz, rows, D, dg):
    """Tiles and sets of views that fill the chip: tiles as deep as the volume, rows
    on the detector and off it.  Of 9e7 samples a few lie so close to the first or
    the last row that a float cannot tell the side; their voxels are left out."""
    _compare(ctx, oracle, 128, 120, nz, 0.5, D, dg, 0.9, rows, 180, edge=2e-6)


@pytest.mark.parametrize("nz", [7, 8, 9, 46])
@pytest.mark.parametrize("views", [2, 7])
def test_few_views(ctx, oracle, nz, views):
    """A chip that they do not fill: tiles of at most 8 slices."""
    _compare(ctx, oracle, 40, 20, nz, 1.0, 200.0, 0.0016, 1.1, 30, views)


def _off_edges(g, xi, beta, D, rz, edge):
    """Voxels none of whose samples lies within edge of the first or last row (64 bits)."""
    nz, ns, nt = g.nz, g.ns, g.nt
    x, y = np.arange(nt) + 0.5 - nt / 2, (np.arange(ns) + 0.5 - ns / 2)[:, None]
    z = ((np.arange(nz) + 0.5 - nz / 2) * rz)[:, None, None]
    keep = np.ones((nz, ns, nt), bool)
    for b in beta:
        u, s = x * np.cos(b) + y * np.sin(b), -x * np.sin(b) + y * np.cos(b)
        r = (2 * D * z / np.hypot(u, D - s) - xi[0]) / (xi[1] - xi[0])
        keep &= (np.abs(r) > edge) & (np.abs(r - (len(xi) - 1)) > edge)
    return keep.ravel()


def _compare(ctx, oracle, nt, ns, nz, rz, D, dg, dx, rows, views, edge=None):
    import ctr
    half = 0.62 * np.hypot(nt, ns)
    n = int(2 * np.arcsin(half / D) / dg) + 2
    gamma = dg * (np.arange(n) - 0.5 * (n - 1) + 0.2)
    xi = dx * (np.arange(rows) - 0.5 * (rows - 1) + 0.1)
    fan = abs(gamma[-1] - gamma[0])
    beta = 0.02 + (np.pi + fan) / views * np.arange(views)
    a = (nt, ns, nz, (nt * 1.0, ns * 1.0, nz * rz), D, 2 * D, beta, gamma, xi, 0.0, fan)
    g, og = ctr.CurvedGeom(*a), oracle.Curved(*a)
    y = np.random.default_rng(nz + views).random(g.nray).astype(np.float32)
    print(f"[case] curved backprojection {nt}x{ns}x{nz}, {views} views of {rows}x{n}", flush=True)
    vol = ctx.curved_bp(g, y)
    with oracle.interp_mode(1):
        ref = oracle.curved_bp(og, y)
    keep = slice(None)
    if edge:
        keep = _off_edges(g, xi, beta, D, rz, edge)
        assert (~keep).sum() <= 20
    e, m = errs(np.asarray(vol).ravel()[keep], np.asarray(ref).ravel()[keep])
    report(f"curved_tiles[{nt}x{ns}x{nz},{n}x{rows}]", rel_l2=e, max_rel=m)
    assert e < 2e-5 and m < 2e-4
    np.testing.assert_array_equal(ctx.curved_bp(g, y, out=vol.copy(), flags=ctr.ACCUMULATE), vol + vol)
