"""The fan adjoint's paths at the sizes where they end: ragged pixel tiles,
fewer views than a block's waves, detectors of either order, rays along the
pixel faces, views with more rays per pixel or per tile than the LDS holds, and
geometries whose ray records are not kept in a table.

Tolerance: a length is an FP64 difference rounded to float once and a pixel's
sum is one float fma chain over n terms, so its error is below n 2^-24 of the
sum of magnitudes (all data are positive here): 1e-5 holds for every n below 160,
and the rms of the chain is far below its bound."""
import numpy as np
import pytest

from conftest import errs, report

pytestmark = pytest.mark.gpu


def geometry(name):
    d = dict(nt=20, ns=17, pixel=1.0, D=60.0, views=25, p=0.6 * (np.arange(70) - 34.5))
    if name == "tile":
        d.update(nt=8, ns=8)
    elif name == "one_pixel":
        d.update(nt=1, ns=1, views=3)
    elif name == "few_views":
        d.update(views=7, nt=33, ns=9)
    elif name == "descending":
        d.update(p=d["p"][::-1].copy())
    elif name == "on_faces":      # odd bins, even pixels: the central ray runs along the faces at four views
        d.update(nt=16, ns=16, views=8, p=0.5 * (np.arange(41) - 20.0))
    elif name == "equiangular":
        d.update(p=60.0 * np.tan(0.012 * (np.arange(61) - 30.0)))
    elif name == "many_per_pixel":   # slots overflow
        d.update(p=0.1 * (np.arange(420) - 209.5))
    elif name == "many_per_tile":    # the staged rays overflow first: 8 pixels of 5 bins
        d.update(p=0.22 * (np.arange(190) - 94.5))
    elif name == "wide_fan":
        d.update(D=13.5, p=13.5 * np.tan(np.linspace(-1.35, 1.35, 90)))
    elif name == "one_bin":
        d.update(p=np.array([0.3]))
    return d


@pytest.mark.parametrize("name", ["base", "tile", "one_pixel", "few_views", "descending", "many_per_pixel", "many_per_tile",
                                  "wide_fan", "one_bin"])
def test_fan_adjoint_paths(ctx, oracle, name):
    import ctr
    d = geometry(name)
    beta = 2 * np.pi / d["views"] * np.arange(1, d["views"] + 1)
    size = (d["nt"] * d["pixel"], d["ns"] * d["pixel"])
    args = (d["nt"], d["ns"], size, d["D"], beta, d["p"])
    g, og = ctr.FanGeom(*args), oracle.Fan(*args)
    y = np.random.default_rng(11).random(g.nray).astype(np.float32)
    print(f"[case] fan adjoint {name}", flush=True)
    e, m = errs(ctx.fan_bp_adjoint(g, y), oracle.fan_adjoint(og, y))
    report(f"fan_adjoint[{name}]", rel_l2=e, max_rel=m)
    assert e < 1e-5 and m < 1e-5


@pytest.mark.parametrize("name", ["on_faces", "equiangular"])
def test_fan_adjoint_rays_on_faces(ctx, oracle, name):
    """Detectors whose central ray runs along pixel faces in some views.  A ray along the pixel faces belongs to the pixels on one side of it
    (which side is a matter of rounding): nothing of it is lost or counted
    twice, so the image sums to the rays' chords."""
    import ctr
    d = geometry(name)
    beta = 2 * np.pi / d["views"] * np.arange(1, d["views"] + 1)
    args = (d["nt"], d["ns"], (float(d["nt"]), float(d["ns"])), d["D"], beta, d["p"])
    g, og = ctr.FanGeom(*args), oracle.Fan(*args)
    y = np.random.default_rng(11).random(g.nray).astype(np.float32)
    total, want = ctx.fan_bp_adjoint(g, y).astype(np.float64).sum(), oracle.fan_adjoint(og, y).sum()
    assert abs(total - want) < 1e-5 * want


def test_fan_adjoint_without_record_table(ctx):
    """More than 2^26 rays: the records are formed by the kernel.  With data in
    60 of 33000 views only, the other views add exact zeros, so the image is
    that of the 60 views alone (whose records are a table) up to a rounding of
    single lengths (an FP64 tail that falls on the other side of a float: at
    most 2^-24 of a term)."""
    import ctr
    import torch
    views, bins, lo, hi = 33000, 2048, 1000, 1060
    beta = 2 * np.pi / views * np.arange(1, views + 1)
    p = 0.02 * (np.arange(bins) - (bins - 1) / 2)
    y = torch.zeros(views, bins, device="cuda")
    y[lo:hi] = torch.rand(hi - lo, bins, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3))
    full = ctx.fan_bp_adjoint(ctr.FanGeom(9, 8, (9.0, 8.0), 30.0, beta, p), y.reshape(-1)).cpu().numpy()
    part = ctx.fan_bp_adjoint(ctr.FanGeom(9, 8, (9.0, 8.0), 30.0, beta[lo:hi], p),
                              y[lo:hi].contiguous().reshape(-1)).cpu().numpy()
    e, m = errs(full, part)
    report("fan_adjoint[no table]", rel_l2=e, max_rel=m)
    assert part.min() > 0 and e < 1e-6 and m < 1e-6


def test_fan_adjoint_ignores_samples_it_does_not_meet(ctx):
    """An infinite sample stays out of the pixels that its ray misses."""
    import ctr
    beta = 2 * np.pi / 12 * np.arange(1, 13)
    p = 0.5 * (np.arange(60) - 29.5)
    g = ctr.FanGeom(24, 24, (24.0, 24.0), 60.0, beta, p)
    y = np.random.default_rng(5).random(g.nray).astype(np.float32)
    a = ctx.fan_bp_adjoint(g, y)
    hit = ctx.fan_bp_adjoint(g, np.eye(1, g.nray, 3 * 60 + 22, dtype=np.float32).ravel()) != 0
    y[3 * 60 + 22] = np.inf
    b = ctx.fan_bp_adjoint(g, y)
    assert hit.any() and not hit.all()
    assert np.all(np.isinf(b[hit])) and np.array_equal(b[~hit], a[~hit])


def test_fan_adjoint_captured_before_its_first_use(ctx):
    """A geometry that only the projector has seen: the captured adjoint allocates
    and waits for nothing, and replays give the eager call's bits, also after the
    eager call has formed the ray records."""
    import ctr
    import torch
    g = ctr.FanGeom(40, 36, (40.0, 36.0), 90.0, 2 * np.pi / 31 * np.arange(31), 0.7 * (np.arange(81) - 40.2))
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        y = ctx.fan_fp(g, torch.rand(g.nvox, device="cuda"))
        out = torch.empty(g.nvox, device="cuda")
        stream.synchronize()
        print("[case] capture", flush=True)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            ctx.fan_bp_adjoint(g, y, out=out)
        for _ in range(3):
            y.copy_(torch.rand(g.nray, device="cuda"))
            out.fill_(float("nan"))
            graph.replay()
            got = out.clone()
            assert torch.equal(got, ctx.fan_bp_adjoint(g, y))
    torch.cuda.synchronize()
    ctx.fan_bp_adjoint(g, np.ones(g.nray, np.float32))


@pytest.mark.parametrize("views", [1, 2, 3, 4, 5, 8, 9])
@pytest.mark.parametrize("name", ["base", "many_per_pixel", "descending"])
def test_fan_adjoint_of_few_views(ctx, oracle, name, views):
    """Blocks of as many waves as views, and the first rounds of whole blocks."""
    import ctr
    d = geometry(name)
    args = (33, 9, (33.0, 9.0), d["D"], 0.4 + 2 * np.pi / views * np.arange(views), d["p"])
    g, og = ctr.FanGeom(*args), oracle.Fan(*args)
    y = np.random.default_rng(views).random(g.nray).astype(np.float32)
    print(f"[case] fan adjoint {name}, {views} views", flush=True)
    e, m = errs(ctx.fan_bp_adjoint(g, y), oracle.fan_adjoint(og, y))
    report(f"fan_adjoint[{name},{views} views]", rel_l2=e, max_rel=m)
    assert e < 1e-5 and m < 1e-5
