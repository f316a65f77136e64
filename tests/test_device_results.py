"""Device-pointer calls on new buffers: every operator writes every element of
its result (the binding does not clear it first), and calls issued one after
the other without a wait between them, on changing inputs and geometries,
give the results of the synchronous host calls bit for bit."""
import numpy as np
import pytest

import ctr

pytestmark = pytest.mark.gpu


def _operators(ctx):
    gc = ctr.geometry.cone_circular(20, 1.0, 14, 41, 33, 1.0, 150.0, 300.0)
    gd = ctr.geometry.cone_circular(33, 1.0, 9, 29, 18, 1.0, 150.0, 300.0)          # truncated
    gf = ctr.geometry.fan_flat(37, 1.0, 13, 50, 1.0, 100.0, 200.0)
    ge = ctr.geometry.fan_equiangular(30, 1.0, 17, 63, 1.0, 100.0, 200.0)
    gp = ctr.ParGeom(35, 22, (35.0, 22.0), np.deg2rad(np.arange(1, 61, 7.0)), np.arange(-14, 14.5, 0.75))
    gam = 0.004 * (np.arange(101) - 50.2)
    gu = ctr.CurvedGeom(24, 20, 9, (24.0, 20.0, 9.0), 90.0, 180.0, 0.21 * np.arange(18), gam,
                        1.1 * (np.arange(15) - 7.0), 0.0, gam[-1] - gam[0])
    for g in (gc, gd):
        yield ctx.cone_fp, g, g.nvox, (), {}
        for f in (ctx.cone_bp_ref, ctx.cone_bp_adjoint, ctx.cone_filter, ctx.fdk_bp, ctx.fdk):
            yield f, g, g.nray, (), {}
        yield ctx.fdk, g, g.nray, (), {"flags": ctr.REF_QUIRKS}
    for g, det in ((gf, ctr.FAN_FLAT), (ge, ctr.FAN_EQUIANGULAR)):
        yield ctx.fan_fp, g, g.nvox, (), {}
        yield ctx.fan_bp_adjoint, g, g.nray, (), {}
        yield ctx.fan_filter, g, g.nray, (det,), {}
        yield ctx.fan_fbp, g, g.nray, (det,), {}
    yield ctx.fan_bp_ref, gf, gf.nray, (), {}
    yield ctx.par_fp, gp, gp.nvox, (), {}
    for f in (ctx.par_bp_adjoint, ctx.par_filter, ctx.par_fbp):
        yield f, gp, gp.nray, (), {}
    for f in (ctx.curved_filter, ctx.curved_bp, ctx.curved_fdk):
        yield f, gu, gu.nray, (), {}
    a = ctr.geometry.iterative_fdk_args(16, n_views=24, pint=2.0)
    yield ctx.fdk_error_slice, ctr.FdkErrGeom(16, 16, 16, a["size"], a["D"], a["beta"], a["u"], a["p"], a["g"], 5), \
        16 ** 3, (), {}


def test_results_are_written_whole_and_in_order(ctx):
    import torch
    rng = np.random.default_rng(7)
    ops = list(_operators(ctx))
    inputs = [rng.random(n).astype(np.float32) for _, _, n, _, _ in ops]
    host = [f(g, x, *a, **k) for (f, g, _, a, k), x in zip(ops, inputs)]
    device = [torch.from_numpy(x).cuda() for x in inputs]
    for dirty in (False, True):
        got = []
        for (f, g, _, a, k), x, h in zip(ops, device, host):
            out = torch.full((h.size,), float("nan"), device="cuda") if dirty else None
            got.append(f(g, x, *a, out=out, **k))
        torch.cuda.synchronize()
        for (f, _, n, _, k), y, h in zip(ops, got, host):
            np.testing.assert_array_equal(y.cpu().numpy().ravel(), h.ravel(), err_msg=f"{f.__name__} {n} {k}")


def test_accumulating_into_a_new_buffer_starts_from_zero(ctx):
    import torch
    g = ctr.geometry.cone_circular(20, 1.0, 14, 41, 33, 1.0, 150.0, 300.0)
    y = torch.rand(g.nray, device="cuda")
    torch.full((4, g.nvox), float("nan"), device="cuda")   # what an uncleared buffer would likely hold
    a = ctx.fdk_bp(g, y, flags=ctr.ACCUMULATE)
    assert torch.equal(a, ctx.fdk_bp(g, y))


@pytest.fixture
def bare(monkeypatch):
    """A context in which every buffer that a call can do without is refused."""
    monkeypatch.setenv("CTR_FAULT", "spare")
    c = ctr.Context(0)
    yield c
    c.close()


def test_calls_do_without_the_memory_of_their_faster_paths(ctx, bare, monkeypatch):
    """View sets, detector columns and ray records need buffers of their own; a call
    that gets none takes the path without them: the same sums in another order, and
    for the projector the other kernel.  2e-6 is the suite's bound for the
    projector; chains of 90 float terms differ by far less."""
    rng = np.random.default_rng(21)
    gc = ctr.geometry.cone_circular(32, 1.0, 90, 64, 64, 1.0, 150.0, 300.0)
    gf = ctr.geometry.fan_flat(64, 1.0, 60, 120, 1.0, 150.0, 300.0)
    gam = 0.004 * (np.arange(101) - 50.2)
    gu = ctr.CurvedGeom(24, 20, 9, (24.0, 20.0, 9.0), 90.0, 180.0, 0.21 * np.arange(18), gam,
                        1.1 * (np.arange(15) - 7.0), 0.0, gam[-1] - gam[0])
    monkeypatch.setenv("CTR_FP_COLUMNS", "1")
    for name, g, n in (("cone_fp", gc, gc.nvox), ("cone_bp_ref", gc, gc.nray), ("cone_bp_adjoint", gc, gc.nray),
                       ("fdk_bp", gc, gc.nray), ("fdk", gc, gc.nray), ("curved_bp", gu, gu.nray),
                       ("curved_fdk", gu, gu.nray), ("fan_bp_adjoint", gf, gf.nray)):
        print(f"[case] {name}", flush=True)
        x = rng.random(n).astype(np.float32)
        a, b = getattr(ctx, name)(g, x), getattr(bare, name)(g, x)
        assert np.linalg.norm(a - b) < 2e-6 * np.linalg.norm(a), name
        if name != "fan_bp_adjoint":   # formed as they go, the records have the same bits
            assert not np.array_equal(a, b), name   # the other path it is

def test_autotuner_times_what_the_calls_run(ctx):
    """A small volume with many views: the calls split the views over sets of blocks
    (an eighth of the time of one set), and so do the autotuner's runs: its best is
    below twice the time of the whole call."""
    import torch
    g = ctr.geometry.cone_circular(32, 1.0, 120, 64, 64, 1.0, 150.0, 300.0)
    proj, vol = torch.rand(g.nray, device="cuda"), torch.empty(g.nvox, device="cuda")
    tuned = ctr.Context(0)
    try:
        r = tuned.autotune_cone(g)
        for name, call in (("bp_ms", tuned.fdk_bp), ("adj_ms", tuned.cone_bp_adjoint)):
            ms = []
            for _ in range(8):
                a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
                a.record()
                call(g, proj, out=vol)
                b.record()
                torch.cuda.synchronize()
                ms.append(a.elapsed_time(b))
            t = float(np.median(ms))
            print(f"[case] {name} {r[name]} call {t}", flush=True)
            assert min(r[name]) < 2 * t
    finally:
        tuned.close()
