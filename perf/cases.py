"""The library's work as a user's program asks for it, as measurable cases.

A case names one call of the Python binding (`ctr.Context` / `ctr.Cnn`) with
its sizes.  `listed()` holds twelve of them, `draw()` makes more of the same
ranges, `prepare()` makes what a program has in hand before the call (a
geometry, device tensors, the process's one context), `run()` makes the call,
`work()` says what it cannot do without and `exact()` computes the same
outputs in 64 bits with plain torch and numpy.

The data are what the operators meet in use: volumes of random ellipsoids,
their analytic line integrals scaled to a largest value of 4 with the noise
of 1e5 photons per ray, and for the network the activations' scales of a SIRT
step.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "ct-research_amd"))
import ctr  # noqa: E402

I0 = 1e5                 # photons per ray
MAX_INTEGRAL = 4.0       # largest line integral of a scan
N_ELL = 10               # ellipsoids of a phantom

# each operator's largest cost (see _cost) that draw() may reach
_LARGEST = {}


def listed():
    cone = dict(voxel=1.0, sod=600.0, sdd=1200.0, pitch=1.0)
    fan = dict(pixel=1.0, sod=500.0, sdd=1000.0, pitch=1.0)
    return [
        # a 2-D preview or a test image: the smallest call, a handful of launches
        dict(name="fan_fp_64", op="fan_fp", nt=64, ns=64, views=90, bins=96, detector="flat", pixel=1.0, sod=150.0,
             sdd=300.0, pitch=2.0),
        # the 2-D fan scan of the benchmark configurations: 256^2, 360 views, 512 equiangular bins, FBP
        dict(name="fan_fbp_256", op="fan_fbp", nt=256, ns=256, views=360, bins=512, detector="equiangular", filt="RL",
             **fan),
        # the same scan reconstructed by SIRT: forward and transposed projector in turn, with its residual history
        dict(name="sirt2d_256", op="sirt2d", nt=256, ns=256, views=360, bins=512, detector="equiangular", iters=10,
             **fan),
        # parallel-beam FBP of FBP_parallel_GPU.m: 512^2 over 60 mm, 360 views, 730 bins of 1.1 pixel
        dict(name="par_fbp_512", op="par_fbp", nt=512, ns=512, views=360, bins=730, filt="SL", pixel=60.0 / 512,
             pitch=1.1 * 60.0 / 512),
        # forward projection of a small ragged volume: a region of interest, a solver's inner call
        dict(name="cone_fp_60", op="cone_fp", nt=60, ns=52, nz=44, views=45, cols=96, rows=80, voxel=1.0, sod=150.0,
             sdd=300.0, pitch=1.6),
        # forward projection at the large workload's size (512^3 at 0.5 mm, 1024 x 768), a third of its views
        dict(name="cone_fp_512", op="cone_fp", nt=512, ns=512, nz=512, views=240, cols=1024, rows=768, voxel=0.5,
             sod=700.0, sdd=1100.0, pitch=0.8),
        # a quick-look FDK of a down-sampled scan
        dict(name="fdk_64", op="fdk", nt=64, ns=64, nz=64, views=90, cols=128, rows=128, filt="SL", voxel=4.0,
             sod=600.0, sdd=1200.0, pitch=4.0),
        # FDK at the benchmark's size: 256^3, 360 views, 512^2 detector
        dict(name="fdk_256", op="fdk", nt=256, ns=256, nz=256, views=360, cols=512, rows=512, filt="SL", **cone),
        # transposed projector of a ragged mid-size volume: the gradient of a data term
        dict(name="adjoint_150", op="adjoint", nt=150, ns=130, nz=101, views=120, cols=211, rows=173, voxel=1.0,
             sod=400.0, sdd=800.0, pitch=1.6),
        # sparse-view SIRT (256^3, 90 views, 512^2 detector), the loop of the iterative and learned methods
        dict(name="sirt3d_256", op="sirt3d", nt=256, ns=256, nz=256, views=90, cols=512, rows=512, iters=2, **cone),
        # the scanner's short scan: 512 x 512 x 50 voxels, 800 views over 240 degrees, 80 rows x 936 channels
        dict(name="curved_fdk_512", op="curved_fdk", nt=512, ns=512, nz=50, views=800, cols=936, rows=80),
        # loss and gradient of the learned update's network on a training batch of four 64^3 patches
        dict(name="cnn_grad_64", op="cnn_grad", patches=4, nx=64, ny=64, nz=64, border=4),
    ]


# ---------------------------------------------------------------------------
# drawing
# ---------------------------------------------------------------------------

def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(c):
    """A case's size in one number: its share of the operator's largest."""
    op = c["op"]
    if op in ("cone_fp", "sirt3d"):
        return c["views"] * c["cols"] * c["rows"] * (c["nt"] + c["ns"]) * (c.get("iters", 1) + 1)
    if op in ("fdk", "adjoint", "curved_fdk"):
        return c["nt"] * c["ns"] * c["nz"] * c["views"]
    if op == "cnn_grad":
        return c["patches"] * c["nx"] * c["ny"] * c["nz"]
    return c["nt"] * c["ns"] * c["views"] * c.get("iters", 1) + c["views"] * c["bins"] ** 2


def _draw_cone(rng, op, n_lo, n_hi, v_lo, v_hi):
    n = _log_int(rng, n_lo, n_hi)
    c = dict(op=op, nt=n, ns=max(8, round(n * rng.uniform(0.8, 1.0))), nz=max(8, round(n * rng.uniform(0.5, 1.0))))
    c["views"] = _log_int(rng, v_lo, v_hi)
    c["voxel"] = rng.choice((0.5, 1.0, 2.0))
    size = c["nt"] * c["voxel"]
    c["sod"] = round(size * rng.uniform(1.6, 3.0), 1)
    c["sdd"] = round(c["sod"] * rng.uniform(1.5, 2.0), 1)
    c["cols"] = max(16, round(n * rng.uniform(1.2, 2.0)))
    c["rows"] = max(16, round(c["nz"] * rng.uniform(1.2, 2.0)))
    c["pitch"] = round(1.25 * size * c["sdd"] / c["sod"] / c["cols"], 4)
    return c


def _draw_fan(rng, op):
    n = _log_int(rng, 64, 512)
    c = dict(op=op, nt=n, ns=max(8, round(n * rng.uniform(0.8, 1.0))), views=_log_int(rng, 60, 720))
    c["pixel"] = rng.choice((0.5, 1.0))
    size = n * c["pixel"]
    c["bins"] = max(32, round(n * rng.uniform(1.2, 2.5)))
    if op == "par_fbp":
        c["pitch"] = round(1.45 * size / c["bins"], 5)
        return c
    c["sod"] = round(size * rng.uniform(1.6, 3.0), 1)
    c["sdd"] = round(c["sod"] * rng.uniform(1.5, 2.0), 1)
    c["pitch"] = round(1.3 * size * c["sdd"] / c["sod"] / c["bins"], 5)
    c["detector"] = rng.choice(("flat", "equiangular"))
    return c


def _draw(rng):
    op = rng.choice(("fan_fp", "fan_fbp", "sirt2d", "par_fbp", "cone_fp", "cone_fp", "fdk", "fdk", "adjoint", "sirt3d",
                     "curved_fdk", "cnn_grad"))
    if op in ("fan_fp", "fan_fbp", "sirt2d", "par_fbp"):
        c = _draw_fan(rng, op)
        if op in ("fan_fbp", "par_fbp"):
            c["filt"] = rng.choice(("SL", "RL"))
        if op == "sirt2d":
            c["iters"] = rng.randint(2, 10)
        return c
    if op == "cone_fp":
        return _draw_cone(rng, op, 32, 512, 20, 360)
    if op == "fdk":
        c = _draw_cone(rng, op, 32, 384, 40, 400)
        c["filt"] = rng.choice(("SL", "RL"))
        return c
    if op == "adjoint":
        return _draw_cone(rng, op, 32, 192, 20, 180)
    if op == "sirt3d":
        c = _draw_cone(rng, op, 32, 256, 20, 120)
        c["iters"] = rng.randint(1, 3)
        return c
    if op == "curved_fdk":
        return dict(op=op, nt=_log_int(rng, 96, 512), ns=_log_int(rng, 96, 512), nz=rng.randint(9, 64),
                    views=_log_int(rng, 120, 800), cols=_log_int(rng, 200, 936), rows=rng.randint(24, 80))
    return dict(op=op, patches=rng.randint(1, 4), nx=_log_int(rng, 24, 72), ny=_log_int(rng, 24, 72),
                nz=_log_int(rng, 24, 72), border=4)


def draw(rng):
    if not _LARGEST:
        for c in listed():
            _LARGEST[c["op"]] = max(_LARGEST.get(c["op"], 0), _cost(c))
        # the 2-D operators are cheap at every size of the range
        for op in ("fan_fp", "fan_fbp", "sirt2d", "par_fbp"):
            _LARGEST[op] = _cost(dict(op=op, nt=512, ns=512, views=720, bins=1280, iters=10))
        # adjoint: the SIRT case's volume and views
        _LARGEST["adjoint"] = 256 ** 3 * 90
    while True:
        c = _draw(rng)
        if _cost(c) <= _LARGEST[c["op"]]:
            return c


# ---------------------------------------------------------------------------
# geometry: plain arrays (the exact values come from these too)
# ---------------------------------------------------------------------------

def _views(n, total=2 * math.pi):
    return total / n * np.arange(1, n + 1, dtype=np.float64)


def _centred(n, pitch):
    return pitch * (np.arange(n, dtype=np.float64) - (n - 1) / 2.0)


def _arrays(c):
    """(size, beta, positions...) of a case's geometry."""
    op = c["op"]
    if op == "curved_fdk":
        # ImplementUIData.m's scanner with the case's counts over the same fan, rows and arc
        fan = 9.7527e-4 * 935
        gamma = -np.linspace(-fan / 2, fan / 2, c["cols"]).astype(np.float32).astype(np.float64)
        xi = np.linspace(-0.5 * 79 * 0.915, 0.5 * 79 * 0.915, c["rows"])
        start = np.deg2rad(1.5466)
        beta = start + np.deg2rad(240.0 / c["views"]) * np.arange(c["views"])
        return (512.0, 512.0, 23.0), beta, gamma, xi, start, abs(gamma[-1] - gamma[0])
    if op == "par_fbp":
        return ((c["nt"] * c["pixel"], c["ns"] * c["pixel"]), np.deg2rad(np.arange(1, c["views"] + 1) * 360.0 / c["views"]),
                _centred(c["bins"], c["pitch"]))
    if "bins" in c:
        size = (c["nt"] * c["pixel"], c["ns"] * c["pixel"])
        if c["detector"] == "equiangular":
            p = c["sod"] * np.tan(_centred(c["bins"], c["pitch"] / c["sdd"]))
        else:
            p = _centred(c["bins"], c["pitch"] * c["sod"] / c["sdd"])
        return size, _views(c["views"]), p
    iso = c["pitch"] * c["sod"] / c["sdd"]
    size = tuple(n * c["voxel"] for n in (c["nt"], c["ns"], c["nz"]))
    return (size, _views(c["views"]).astype(np.float32), _centred(c["cols"], iso).astype(np.float32),
            _centred(c["rows"], iso).astype(np.float32))


def _geometry(c):
    a = _arrays(c)
    if c["op"] == "curved_fdk":
        size, beta, gamma, xi, start, fan = a
        return ctr.CurvedGeom(c["nt"], c["ns"], c["nz"], size, 570.0, 1060.2, beta, gamma, xi, start, fan)
    if c["op"] == "par_fbp":
        return ctr.ParGeom(c["nt"], c["ns"], *a)
    if "bins" in c:
        return ctr.FanGeom(c["nt"], c["ns"], a[0], c["sod"], a[1], a[2])
    return ctr.ConeGeom(c["nt"], c["ns"], c["nz"], a[0], c["sod"], a[1], a[2], a[3])


# ---------------------------------------------------------------------------
# data
# ---------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _ellipsoids(c, size, seed):
    """[(centre (3), inverse semi-axes (3), cos, sin, amplitude)] inside the field of view, mm from the centre."""
    rng = np.random.default_rng(seed)
    a = _arrays(c)
    half = 0.5 * np.array(size if len(size) == 3 else (*size, 1.0))
    if c["op"] == "curved_fdk":
        fov = 570.0 * math.sin(0.5 * a[5])
    elif c["op"] == "par_fbp":
        fov = abs(a[2][-1])
    else:
        fov = c["sod"] * math.sin(math.atan(abs(float(a[2][-1])) / c["sod"]))
    r = 0.85 * min(half[0], half[1], fov)
    rz = 0.85 * half[2] if len(size) == 3 else 1.0
    out = [(np.zeros(3), 1.0 / np.array([0.95 * r, 0.9 * r, rz]), 1.0, 0.0, 1.0)]
    for _ in range(N_ELL - 1):
        ax = np.array([rng.uniform(0.05, 0.35) * r, rng.uniform(0.05, 0.35) * r, rng.uniform(0.1, 0.4) * rz])
        rad, ang = rng.uniform(0, 0.55) * r, rng.uniform(0, 2 * math.pi)
        cen = np.array([rad * math.cos(ang), rad * math.sin(ang), rng.uniform(-0.5, 0.5) * rz])
        phi = rng.uniform(0, math.pi)
        out.append((cen, 1.0 / ax, math.cos(phi), math.sin(phi), rng.uniform(-0.3, 0.5)))
    return out


def _volume(c, size, seed):
    n = (c["nt"], c["ns"], c.get("nz", 1))
    s3 = tuple(size) if len(size) == 3 else (*size, 1.0)
    ax = [torch.from_numpy(((np.arange(n[k]) + 0.5) * s3[k] / n[k] - s3[k] / 2).astype(np.float32)).cuda()
          for k in range(3)]
    x, y, z = ax[0][None, None, :], ax[1][None, :, None], ax[2][:, None, None]
    vol = torch.zeros(n[2], n[1], n[0], device="cuda")
    for cen, inv, cp, sp, amp in _ellipsoids(c, size, seed):
        u, v = (x - cen[0]) * cp + (y - cen[1]) * sp, (y - cen[1]) * cp - (x - cen[0]) * sp
        q = (u * inv[0]) ** 2 + (v * inv[1]) ** 2
        inside = q + (((z - cen[2]) * inv[2]) ** 2 if len(size) == 3 else 0.0) <= 1.0
        vol.add_(inside, alpha=float(amp))
    # texture, as reconstructed volumes have
    vol += 0.01 * torch.randn(vol.shape, device="cuda", generator=_gen(seed))
    return vol.reshape(-1)


def _chord(S, d, e, three):
    """Chord length of the rays S + l d (d of unit length) through ellipsoid e."""
    cen, inv, cp, sp, amp = e
    ox, oy = S[0] - cen[0], S[1] - cen[1]
    a0, a1 = (ox * cp + oy * sp) * inv[0], (oy * cp - ox * sp) * inv[1]
    b0, b1 = (d[0] * cp + d[1] * sp) * inv[0], (d[1] * cp - d[0] * sp) * inv[1]
    A, B, C = b0 * b0 + b1 * b1, a0 * b0 + a1 * b1, a0 * a0 + a1 * a1 - 1.0
    if three:
        a2, b2 = (S[2] - cen[2]) * inv[2], d[2] * inv[2]
        A, B, C = A + b2 * b2, B + a2 * b2, C + a2 * a2
    return 2.0 * amp * torch.sqrt(torch.clamp(B * B - A * C, min=0.0)) / A


def _projections(c, seed):
    """Analytic line integrals of the phantom, scaled to a largest value of 4, with photon noise."""
    a = _arrays(c)
    size, beta = a[0], a[1]
    three = len(size) == 3
    ells = _ellipsoids(c, size, seed)
    gen = _gen(seed)
    f = lambda v: torch.from_numpy(np.ascontiguousarray(v, dtype=np.float32)).cuda()
    rows = len(a[3]) if three else 1
    out = torch.empty(len(beta), rows, len(a[2]), device="cuda")
    step = max(1, (1 << 24) // (rows * len(a[2])))
    for b0 in range(0, len(beta), step):
        bb = beta[b0:b0 + step].astype(np.float64)
        sb, cb = f(np.sin(bb))[:, None, None], f(np.cos(bb))[:, None, None]
        if c["op"] == "par_fbp":
            p = f(a[2])[None, None, :]
            S, d = (p * cb, p * sb), (-sb + 0 * p, cb + 0 * p)
        elif c["op"] == "curved_fdk":
            D, Dsd = 570.0, 1060.2
            gam, xi = f(a[2])[None, None, :], f(a[3])[None, :, None]
            S = (-D * sb, D * cb, 0.0)
            sg, cg = torch.sin(gam), torch.cos(gam)
            d = (sg * cb + cg * sb, sg * sb - cg * cb, xi / Dsd)
        else:
            D, p = c["sod"], f(a[2])[None, None, :]
            S = (-D * sb, D * cb, 0.0)
            d = (p * cb + D * sb, p * sb - D * cb, f(a[3])[None, :, None] if three else None)
        n2 = d[0] * d[0] + d[1] * d[1] + (d[2] * d[2] if three else 0.0)
        inv = torch.rsqrt(n2)
        d = tuple(v * inv for v in d if v is not None)
        acc = torch.zeros(len(bb), rows, len(a[2]), device="cuda")
        for e in ells:
            acc += _chord(S, d, e, three)
        out[b0:b0 + step] = acc
    out.mul_(MAX_INTEGRAL / torch.clamp(out.max(), min=1e-6))
    for b0 in range(0, len(beta), step):
        o = out[b0:b0 + step]
        o += torch.randn(o.shape, device="cuda", generator=gen) * torch.exp(0.5 * o) / math.sqrt(I0)
    return out.reshape(-1)


def prepare(case, seed):
    op = case["op"]
    ctx = ctr.default_context()
    if op == "cnn_grad":
        net = ctr.Cnn(ctx, ctr.cnn_init_params(seed, last_scale=1.0))
        gen = _gen(seed)
        n = (case["patches"], case["nz"], case["ny"], case["nx"])
        x = torch.rand(n, device="cuda", generator=gen)
        g = 0.02 * torch.randn(n, device="cuda", generator=gen)
        t = torch.randn(n, device="cuda", generator=gen)
        return dict(op=op, net=net, shape=(case["nx"], case["ny"], case["nz"]), x=x, g=g, target=t,
                    scale=np.full(case["patches"], 50.0, np.float32), border=case["border"])
    s = dict(op=op, ctx=ctx, geom=_geometry(case), iters=case.get("iters"),
             filt=ctr.FILTER_RL_HALF if case.get("filt") == "RL" else ctr.FILTER_SL_HALF,
             det=ctr.FAN_EQUIANGULAR if case.get("detector") == "equiangular" else ctr.FAN_FLAT)
    s["data"] = _volume(case, _arrays(case)[0], seed) if op in ("fan_fp", "cone_fp") else _projections(case, seed)
    return s


def run(s):
    op = s["op"]
    if op == "cnn_grad":
        loss, grad = s["net"].train_step(s["shape"], s["x"], s["g"], s["scale"], s["target"], border=s["border"],
                                         want_grad=True)
        return {"loss": loss, "grad": grad}
    ctx, g, data = s["ctx"], s["geom"], s["data"]
    if op == "fan_fp":
        return ctx.fan_fp(g, data)
    if op == "fan_fbp":
        return ctx.fan_fbp(g, data, s["det"], s["filt"])
    if op == "par_fbp":
        return ctx.par_fbp(g, data, s["filt"])
    if op == "cone_fp":
        return ctx.cone_fp(g, data)
    if op == "fdk":
        return ctx.fdk(g, data, s["filt"])
    if op == "adjoint":
        return ctx.cone_bp_adjoint(g, data)
    if op == "curved_fdk":
        return ctx.curved_fdk(g, data)
    x, r2, r1 = (ctx.sirt3d if op == "sirt3d" else ctx.sirt2d)(g, data, s["iters"])
    return {"x": x, "residual_l2": r2, "residual_l1": r1}


def work(case):
    op = case["op"]
    if op == "cnn_grad":
        n = case["patches"] * case["nx"] * case["ny"] * case["nz"]
        # multiply-adds of the four layers, forward and both gradients (no input gradient of the first layer)
        macs = 27 * (2 * 32 * 2 + 32 * 32 * 3 * 2 + 32 * 3)
        return {"bytes": 12 * n + 8 * ctr.CNN_NUM_PARAMS, "flops": 2 * macs * n}
    nvox = case["nt"] * case["ns"] * case.get("nz", 1)
    nray = case["views"] * (case["bins"] if "bins" in case else case["cols"] * case["rows"])
    it = case.get("iters", 1)
    seg = 0.7 * (case["nt"] + case["ns"])          # voxels of a mean ray
    upd = nvox * case["views"]
    cols = case.get("bins", case.get("cols", 0))
    filt = nray * 5 * math.log2(max(2, 2 * cols)) * 2
    flops = {"fan_fp": 2 * nray * seg, "cone_fp": 2 * nray * seg, "adjoint": 2 * nray * seg,
             "sirt2d": (2 * it + 1) * 2 * nray * seg, "sirt3d": (2 * it + 1) * 2 * nray * seg,
             "fan_fbp": filt + 8 * upd, "par_fbp": filt + 6 * upd, "fdk": filt + 10 * upd,
             "curved_fdk": filt + 16 * upd}[op]
    passes = 2 * it + 1 if op.startswith("sirt") else 1
    return {"bytes": 4 * (nvox + nray) * passes, "flops": flops}


# ---------------------------------------------------------------------------
# 64 bits, plain torch
# ---------------------------------------------------------------------------

def _d(v):
    return torch.from_numpy(np.ascontiguousarray(v, dtype=np.float64)).cuda()


class _Siddon:
    """The ray-driven projector A and its transpose, one crossing at a time."""

    def __init__(self, case):
        a = _arrays(case)
        self.three = len(a[0]) == 3
        self.n = (case["nt"], case["ns"], case.get("nz", 1))
        self.size = tuple(a[0]) if self.three else (*a[0], 1.0)
        self.r = tuple(s / n for s, n in zip(self.size, self.n))
        self.D = case["sod"]
        self.beta, self.p = a[1].astype(np.float64), _d(a[2])
        self.xi = _d(a[3]) if self.three else _d([0.0])
        self.per_view = self.p.numel() * self.xi.numel()
        self.nray = self.per_view * len(self.beta)
        self.nvox = self.n[0] * self.n[1] * self.n[2]
        self.chunk = max(1, (1 << 22) // self.per_view)

    def _walk(self, visit, lo_view, hi_view):
        b = self.beta[lo_view:hi_view]
        sb, cb = _d(np.sin(b))[:, None, None], _d(np.cos(b))[:, None, None]
        p, xi = self.p[None, None, :], self.xi[None, :, None]
        zero = torch.zeros(len(b), self.xi.numel(), self.p.numel(), dtype=torch.float64, device="cuda")
        d = [p * cb + self.D * sb + zero, p * sb - self.D * cb + zero, xi + zero]
        norm = torch.sqrt(d[0] ** 2 + d[1] ** 2 + d[2] ** 2)
        d = [(v / norm).reshape(-1) for v in d]
        S = [(self.size[0] / 2 - self.D * sb + zero).reshape(-1), (self.size[1] / 2 + self.D * cb + zero).reshape(-1),
             (self.size[2] / 2 + zero).reshape(-1)]
        axes = (0, 1, 2) if self.three else (0, 1)
        lo = torch.full_like(S[0], -math.inf)
        hi = torch.full_like(S[0], math.inf)
        for k in axes:
            t1, t2 = -S[k] / d[k], (self.size[k] - S[k]) / d[k]
            flat = d[k] == 0
            inside = (S[k] >= 0) & (S[k] < self.size[k])
            lo = torch.where(flat, torch.where(inside, lo, math.inf), torch.maximum(lo, torch.minimum(t1, t2)))
            hi = torch.where(flat, hi, torch.minimum(hi, torch.maximum(t1, t2)))
        hit = hi > lo
        lo, hi = torch.where(hit, lo, 0.0), torch.where(hit, hi, 0.0)
        lam = lo
        plane, nxt, idx, strides = [], [], torch.zeros_like(lo, dtype=torch.int64), (1, self.n[0], self.n[0] * self.n[1])
        steps = []
        for k in axes:
            pos = (S[k] + lo * d[k]) / self.r[k]
            up = d[k] > 0
            i = torch.where(up, torch.floor(pos), torch.ceil(pos) - 1).clamp(0, self.n[k] - 1)
            idx = idx + i.to(torch.int64) * strides[k]
            pl = torch.where(up, i + 1, i)
            plane.append(pl)
            nxt.append(torch.where(d[k] == 0, math.inf, (pl * self.r[k] - S[k]) / d[k]))
            steps.append(torch.where(up, 1.0, -1.0))
        top = self.nvox - 1
        for it in range(sum(self.n) + 3):
            m = hi
            for v in nxt:
                m = torch.minimum(m, v)
            visit(idx.clamp(0, top), torch.clamp(m - lam, min=0.0))
            lam = torch.maximum(m, lam)
            for q, k in enumerate(axes):
                go = nxt[q] <= m
                plane[q] = plane[q] + torch.where(go, steps[q], 0.0)
                nxt[q] = torch.where(go, (plane[q] * self.r[k] - S[k]) / d[k], nxt[q])
                idx = idx + torch.where(go, steps[q], 0.0).to(torch.int64) * strides[k]
            if it % 16 == 15 and not bool((lam < hi).any()):
                break

    def _chunks(self):
        for v in range(0, len(self.beta), self.chunk):
            w = min(v + self.chunk, len(self.beta))
            yield v, w, slice(v * self.per_view, w * self.per_view)

    def forward(self, x):
        """(A x, A 1)"""
        ax = torch.zeros(self.nray, dtype=torch.float64, device="cuda")
        rows = torch.zeros_like(ax)
        for v, w, sl in self._chunks():
            a, r = ax[sl], rows[sl]

            def visit(idx, length):
                a.addcmul_(length, x[idx])
                r.add_(length)
            self._walk(visit, v, w)
        return ax, rows

    def transpose(self, y):
        out = torch.zeros(self.nvox, dtype=torch.float64, device="cuda")
        for v, w, sl in self._chunks():
            yy = y[sl]
            self._walk(lambda idx, length: out.index_add_(0, idx, length * yy), v, w)
        return out


def _sirt(A, b, iters):
    cols = A.transpose(torch.ones_like(b))
    x = torch.zeros(A.nvox, dtype=torch.float64, device="cuda")
    r2, r1 = [], []
    for k in range(iters + 1):
        ax, rows = A.forward(x)
        e = b - ax
        r2.append(float(e.norm() / b.norm()))
        r1.append(float(e.abs().sum() / (b.sum() * A.nvox)))
        if k < iters:
            x = torch.clamp(x + A.transpose(e / (rows + 1e-9)) / (cols + 1e-9), min=0.0)
    return {"x": x, "residual_l2": np.array(r2), "residual_l1": np.array(r1)}


def _taps(filt, d, n, equiangular=False):
    """Half-scaled ramp taps; the Shepp-Logan ones are stored in single precision by definition."""
    k = np.arange(n, dtype=np.float64)
    if filt == "SL":
        return (-1.0 / (d * np.pi) ** 2 / (4 * k * k - 1)).astype(np.float32).astype(np.float64)
    h = np.zeros(n)
    h[0] = 1.0 / (8 * d * d)
    odd = slice(1, None, 2)
    h[odd] = -1.0 / (2 * np.pi ** 2 * (np.sin(k[odd] * d) ** 2 if equiangular else k[odd] ** 2 * d * d))
    return h


def _convolve(rows, taps):
    """rows [..., n] with the even kernel taps [..., n]."""
    n = rows.shape[-1]
    L = 1 << (2 * n - 1).bit_length()
    ker = torch.zeros(*taps.shape[:-1], L, dtype=torch.float64, device="cuda")
    ker[..., :n] = taps
    ker[..., L - n + 1:] = taps[..., 1:].flip(-1)
    return torch.fft.irfft(torch.fft.rfft(rows, L) * torch.fft.rfft(ker), L)[..., :n]


def _sample(rows, u):
    """Linear samples of rows [n] at u, 0 outside [0, n - 1)."""
    ok = (u >= 0) & (u < rows.shape[-1] - 1)
    i = u.floor().clamp(0, rows.shape[-1] - 2)
    f = u - i
    i = i.to(torch.int64)
    return torch.where(ok, rows[i] * (1 - f) + rows[i + 1] * f, 0.0)


def _bilinear(img, u, v):
    """Bilinear samples of img [rows, cols] at (u, v), 0 outside [0, cols - 1) x [0, rows - 1)."""
    nr, nc = img.shape
    ok = (u >= 0) & (u < nc - 1) & (v >= 0) & (v < nr - 1)
    grid = torch.stack((u * (2.0 / (nc - 1)) - 1, v * (2.0 / (nr - 1)) - 1), dim=-1)
    s = torch.nn.functional.grid_sample(img[None, None], grid.reshape(1, 1, -1, 2), align_corners=True)
    return torch.where(ok, s.reshape(u.shape), 0.0)


def _pixels(case, size):
    x = _d((np.arange(case["nt"]) + 0.5) * size[0] / case["nt"] - size[0] / 2)[None, :]
    y = _d((np.arange(case["ns"]) + 0.5) * size[1] / case["ns"] - size[1] / 2)[:, None]
    return x, y


def _grid(pos):
    """(first, step) of the uniform grid through the end samples."""
    pos = np.asarray(pos, np.float64)
    return pos[0], (pos[-1] - pos[0]) / (len(pos) - 1)


def _exact_fdk(case, data):
    size, beta, p, xi = _arrays(case)
    D, nb, nr, nc = case["sod"], len(beta), len(xi), len(p)
    pd, xd = _d(p)[None, :], _d(xi)[:, None]
    w = D / torch.sqrt(D * D + pd * pd + xd * xd)
    d = float(abs(p[1] - p[0]))
    taps = _d(_taps(case["filt"], d, nc) * d)
    x, y = _pixels(case, size)
    z = _d((np.arange(case["nz"]) + 0.5) * size[2] / case["nz"] - size[2] / 2)[:, None, None]
    (p0, dp), (x0, dx) = _grid(p), _grid(xi)
    vol = torch.zeros(case["nz"], case["ns"], case["nt"], dtype=torch.float64, device="cuda")
    for b in range(nb):
        # the weighted samples are stored in single precision by definition
        q = _convolve((data.reshape(nb, nr, nc)[b].double() * w).float().double(), taps)
        sb, cb = math.sin(float(beta[b])), math.cos(float(beta[b]))
        m = D / (D - (-x * sb + y * cb))
        u = ((x * cb + y * sb) * m - p0) / dp
        v = (z * m - x0) / dx
        vol += _bilinear(q, u.expand_as(v), v) * (m * m)
    return (vol * float(abs(beta[1] - beta[0]))).reshape(-1)


def _exact_curved(case, data):
    size, beta, gamma, xi, start, fan = _arrays(case)
    D, Dsd, pi = 570.0, 1060.2, math.pi
    nb, nr, nc = len(beta), len(xi), len(gamma)
    P = Dsd / np.sqrt(Dsd * Dsd + xi * xi)
    dg = abs(gamma[1] - gamma[0])
    k = np.arange(nc, dtype=np.float64)[None, :]
    dgp = (dg * P)[:, None]
    with np.errstate(divide="ignore", invalid="ignore"):
        taps = -2 * k * k / (pi * pi) / (4 * k * k - 1) / np.sin(k * dgp) ** 2
    taps[:, 0] = 2 / (pi * dgp[:, 0]) ** 2
    taps = _d(taps * dgp)
    g, Pd = _d(gamma)[None, :] * _d(P)[:, None], _d(P)[:, None]
    x, y = _pixels(case, size)
    z = _d((np.arange(case["nz"]) + 0.5) * size[2] / case["nz"] - size[2] / 2)[:, None, None]
    (g0, gs), (x0, dx) = _grid(gamma), _grid(xi)
    vol = torch.zeros(case["nz"], case["ns"], case["nt"], dtype=torch.float64, device="cuda")
    for b in range(nb):
        bp, st, fp = float(beta[b]) * Pd, start * Pd, fan * Pd
        up = (bp >= st) & (bp < st + fp - 2 * g)
        flat = (bp >= st + fp - 2 * g) & (bp <= st + pi - 2 * g)
        down = (bp > st + pi - 2 * g) & (bp <= st + pi + fp)
        d1, d2 = fp / 2 - g, fp / 2 + g
        w1 = torch.where(d1 > 0, torch.sin(pi / 4 * bp / d1) ** 2, 0.0)
        w2 = torch.where(d2 > 0, torch.sin(pi / 4 * (pi + fp - bp) / d2) ** 2, 0.0)
        park = torch.where(up, w1, torch.where(flat, 1.0, torch.where(down, w2, 0.0)))
        q = _convolve(data.reshape(nb, nr, nc)[b].double() * (D / Pd) * torch.cos(g) * park, taps)
        sb, cb = math.sin(beta[b]), math.cos(beta[b])
        u, ds = x * cb + y * sb, D - (-x * sb + y * cb)
        rho2 = u * u + ds * ds
        L2 = rho2 + z * z
        v = (Dsd * z / torch.sqrt(rho2) - x0) / dx
        c = (torch.atan(u / ds) - g0) / gs
        vol += _bilinear(q, c.expand_as(v), v) * (torch.sqrt(rho2) / (L2 * torch.sqrt(L2)))
    return (vol * abs(beta[1] - beta[0])).reshape(-1)


def _exact_2d(case, data):
    size, beta, p = _arrays(case)
    nb, nc = len(beta), len(p)
    rows = data.reshape(nb, nc).double()
    x, y = _pixels(case, size)
    img = torch.zeros(case["ns"], case["nt"], dtype=torch.float64, device="cuda")
    if case["op"] == "fan_fbp" and case["detector"] == "equiangular":
        D = case["sod"]
        gam = np.arctan(p / D)
        d = abs(gam[1] - gam[0])
        q = _convolve(rows * _d(D * np.cos(gam)), _d(_taps("RL", d, nc, True) * d if case["filt"] == "RL" else
                                                    -1.0 / (d * np.pi) ** 2 / (4 * np.arange(nc) ** 2.0 - 1) * d))
        g0, dg = _grid(gam)
        for b in range(nb):
            sb, cb = math.sin(beta[b]), math.cos(beta[b])
            u, w = x * cb + y * sb, D - (-x * sb + y * cb)
            img += _sample(q[b], (torch.atan2(u, w) - g0) / dg) / (u * u + w * w)
        return (img * abs(beta[1] - beta[0])).reshape(-1)
    pf = p.astype(np.float32).astype(np.float64)
    bf = beta.astype(np.float32).astype(np.float64)
    d = float(abs(np.float32(p[1]) - np.float32(p[0])))
    taps = _d(_taps(case["filt"], d, nc) * d)
    p0, dp = _grid(pf)
    if case["op"] == "par_fbp":
        q = _convolve(rows, taps)
        for b in range(nb):
            img += _sample(q[b], (x * math.cos(bf[b]) + y * math.sin(bf[b]) - p0) / dp)
    else:
        D = case["sod"]
        w = _d(D / np.sqrt(D * D + pf * pf))
        q = _convolve((rows * w).float().double(), taps)
        for b in range(nb):
            sb, cb = math.sin(beta[b]), math.cos(beta[b])
            U = (D - (-x * sb + y * cb)) / D
            img += _sample(q[b], ((x * cb + y * sb) / U - p0) / dp) / (U * U)
    return (img * abs(bf[1] - bf[0])).reshape(-1)


def _exact_cnn(case, seed):
    s = prepare(case, seed)
    params = torch.from_numpy(ctr.cnn_init_params(seed, last_scale=1.0)).double().cuda().requires_grad_(True)
    nx, ny, nz = s["shape"]
    n, b = case["patches"], case["border"]
    total = 0.0
    for i in range(n):
        h = torch.stack((s["x"][i], s["g"][i] * float(s["scale"][i]))).double()
        o = 0
        for li, (co, ci) in enumerate(((32, 2), (32, 32), (32, 32), (1, 32))):
            w = params[o:o + co * ci * 27].reshape(co, ci, 3, 3, 3)
            bias = params[o + co * ci * 27:o + co * ci * 27 + co]
            o += co * ci * 27 + co
            pad = torch.nn.functional.pad(h, (1,) * 6)
            out = bias[:, None].expand(co, nz * ny * nx)
            for t in range(27):
                dz, dy, dx = t // 9, t // 3 % 3, t % 3
                out = out + w[:, :, dz, dy, dx] @ pad[:, dz:dz + nz, dy:dy + ny, dx:dx + nx].reshape(ci, -1)
            h = out.reshape(co, nz, ny, nx)
            if li < 3:
                h = torch.relu(h)
        e = (h[0] - s["target"][i].double())[b:nz - b, b:ny - b, b:nx - b]
        loss = e.square().mean() / n
        loss.backward()
        total += float(loss)
    return {"loss": total, "grad": params.grad.detach()}


def exact(case, seed):
    op = case["op"]
    if op == "cnn_grad":
        return _exact_cnn(case, seed)
    if op in ("fan_fp", "cone_fp", "adjoint", "sirt2d", "sirt3d"):
        # crossings of all rays and passes, walked here at 1e9 to 7e9 a second (the transpose is the slower)
        nray = case["views"] * (case["bins"] if "bins" in case else case["cols"] * case["rows"])
        sweeps = 2 * case["iters"] + 2 if "iters" in case else 1
        if nray * (case["nt"] + case["ns"]) * sweeps > 2e10:
            return None
        s = prepare(case, seed)
        A, data = _Siddon(case), s["data"].double()
        if op in ("fan_fp", "cone_fp"):
            return A.forward(data)[0]
        if op == "adjoint":
            return A.transpose(data)
        return _sirt(A, data, case["iters"])
    data = prepare(case, seed)["data"]
    if op == "fdk":
        return _exact_fdk(case, data)
    if op == "curved_fdk":
        return _exact_curved(case, data)
    return _exact_2d(case, data)
