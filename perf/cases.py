"""The work a user of this framework has it do, as timed cases.

Each case is one call (or one forward and backward) through the public entry
points, at sizes between a single ray and the largest workloads the
benchmark runs:

  single     core.single_ray on host numbers
  tracing    core.ray_tracing on host arrays, a Dataset back (the drop-in call)
  device     core.trace_many_device on device tensors, into kept outputs
  gradient   adjoint.trace_differentiable and its backward pass
  iteration  one descent iteration of the current inversion: forward with
             checkpoints, residuals, reverse sweep
  batch      Batch.run: many scenes in one persistent launch

and by the fields the rays cross:

  shared     depth and current on one grid (one ocean model's output)
  separate   depth and current on grids of their own (a chart and a model)
  depth      gridded depth under a constant current
  current    gridded current over a constant depth
  slope      a plane beach under a constant current (no grid)

listed() names the cases, draw() gives more of the same ranges, prepare()
makes what a program holds before the call, run() is one pass, work() what
the path cannot do without, and exact() the outputs in 64 bits from plain
torch operations.
"""
from __future__ import annotations

import math

import torch

from mantaray_amd import adjoint, core
from mantaray_amd.batch import Batch
from mantaray_amd.fields import Bathymetry, Current

G = 9.8
STATE = ("x", "y", "kx", "ky")
FLOP_PER_RAY_STEP = 745       # 265 basic f64 operations and 24 transcendentals x 20
DEV = "cuda:0"

_DEFAULTS = {"entry": "device", "fields": "shared", "bed": "seamount", "nx": 501, "ny": 501,
             "dx": 200.0, "ratio": 2.7, "scenes": 1, "rays": 1000, "steps": 500, "dt": 1.0,
             "math": "fast", "precision": "reference", "solout": "state", "rows": False,
             "stride": 50}


def _case(name=None, **kw):
    c = {**_DEFAULTS, **kw}
    return {"name": name, **c} if name else c


def listed():
    return [
        # one ray through a model's output: the call of a notebook or a quick look
        _case("single ray", entry="single", bed="shelf", rays=1, steps=1000, dx=100.0, rows=True),
        # the reference's own example size: a fan of rays up a beach, host in and out
        _case("beach fan, host", entry="tracing", bed="shelf", rays=128, steps=1000, dx=100.0,
              rows=True),
        # a study of many rays through the drop-in call, a chart and a current
        # model on their own grids; the answer is 260 MB on the host
        _case("study, host", entry="tracing", fields="separate", bed="shelf", nx=613, ny=409,
              rays=8191, steps=1000, rows=True),
        # a small device call inside a larger program (a few rays, end states)
        _case("few rays, short", rays=257, steps=120, nx=256, ny=256, dt=2.0),
        # the headline workload: full trajectories of 65,536 rays
        _case("seamount jet", nx=1024, ny=1024, rays=65536, steps=5000, rows=True),
        # depth from a chart, current from a coarser model: the usual data
        _case("chart and model", fields="separate", bed="shelf", nx=1201, ny=907, dx=150.0,
              rays=30011, steps=2000, dt=0.7, rows=True),
        # bathymetry only, no current: swell over a shelf, end states
        _case("depth only", fields="depth", bed="shelf", nx=1024, ny=768, rays=20000, steps=1500),
        # the reference's own formulas, where agreement with it comes first
        _case("literal formulas", nx=512, ny=512, rays=16384, steps=500, math="literal",
              rows=True),
        # the differentiable path's workload: a loss on end points, gradients
        # of the launch states and of the current
        _case("eddy gradient", entry="gradient", fields="current", nx=512, ny=512, dx=250.0,
              rays=16384, steps=2000),
        # a loss on whole trajectories, gradients of depth and current too
        _case("depth and current gradient", entry="gradient", fields="shared", bed="shelf",
              nx=401, ny=301, rays=4099, steps=600, rows=True, stride=25),
        # the largest: one iteration of the current inversion
        _case("inversion iteration", entry="iteration", fields="current", nx=2048, ny=2048,
              dx=100.0, rays=262144, steps=3000),
        # an ensemble of scenes of uneven size in one launch
        _case("ensemble", entry="batch", nx=700, ny=700, dx=250.0, scenes=24, rays=98304,
              steps=1500),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    entry = rng.choice(["single", "tracing", "tracing", "device", "device", "device", "device",
                        "gradient", "gradient", "iteration", "batch"])
    c = {"entry": entry, "bed": rng.choice(["shelf", "seamount"]), "nx": _log(rng, 150, 1500),
         "ny": _log(rng, 150, 1500), "dx": float(rng.choice([100, 150, 200, 250, 500])),
         "ratio": rng.choice([1.5, 2.7, 4.0]), "dt": rng.choice([1.0, 1.0, 2.0, 0.5, 0.7])}
    if entry == "single":
        c.update(rays=1, steps=_log(rng, 100, 3000), rows=True,
                 fields=rng.choice(["shared", "separate", "slope"]))
    elif entry == "tracing":
        c.update(rays=_log(rng, 20, 8000), steps=_log(rng, 100, 1500), rows=True,
                 fields=rng.choice(["shared", "separate", "depth", "slope"]))
    elif entry == "device":
        c.update(rays=_log(rng, 200, 100000), steps=_log(rng, 100, 3000),
                 fields=rng.choice(["shared", "shared", "separate", "separate", "depth",
                                    "current", "slope"]),
                 rows=rng.random() < 0.5, solout=rng.choice(["state", "state", "next_deriv"]),
                 math=rng.choice(["fast", "fast", "fast", "literal"]),
                 precision=rng.choice(["reference", "reference", "reference", "fp64"]))
    elif entry == "gradient":
        c.update(rays=_log(rng, 500, 30000), steps=_log(rng, 100, 1500),
                 fields=rng.choice(["current", "shared", "separate"]),
                 rows=rng.random() < 0.4, stride=rng.choice([20, 25, 50, 64]))
    elif entry == "iteration":
        c.update(rays=_log(rng, 20000, 200000), steps=_log(rng, 300, 1500),
                 fields=rng.choice(["current", "current", "shared"]))
    else:
        c.update(scenes=rng.randint(6, 40), rays=_log(rng, 10000, 150000),
                 steps=_log(rng, 300, 2500), fields=rng.choice(["shared", "shared", "separate"]),
                 nx=_log(rng, 200, 800), ny=_log(rng, 200, 800))
    return _case(**c)


# ---------------------------------------------------------------------------
# inputs, from the seed alone

def _axis(n, dx):
    return torch.arange(n, dtype=torch.float64, device=DEV) * dx


def _depth(g, x, y, bed):
    """Depth [ny, nx]: a seamount in deep water, or a shelf that shoals along
    x with banks and troughs on it."""
    lx, ly = float(x[-1]), float(y[-1])
    if bed == "seamount":
        xc, yc = (float(v) for v in 0.4 + 0.2 * torch.rand(2, generator=g, dtype=torch.float64))
        s = 0.075 * min(lx, ly)
        r2 = (x[None, :] - xc * lx) ** 2 + (y[:, None] - yc * ly) ** 2
        return 4000.0 - 3800.0 * torch.exp(-r2 / (2.0 * s * s))
    d = (180.0 - 150.0 * (x / lx))[None, :].expand(y.numel(), x.numel()).clone()
    for xc, yc, s, a in torch.rand((12, 4), generator=g, dtype=torch.float64).tolist():
        s = (0.04 + 0.08 * s) * min(lx, ly)
        d += (a - 0.6) * 30.0 * torch.outer(torch.exp(-(y - yc * ly) ** 2 / (2 * s * s)),
                                            torch.exp(-(x - xc * lx) ** 2 / (2 * s * s)))
    return d.clamp_(min=2.0)


def _eddies(g, x, y):
    """u, v [ny, nx]: a zonal jet and twelve Gaussian eddies."""
    lx, ly = float(x[-1]), float(y[-1])
    u = (0.8 / torch.cosh((y - 0.5 * ly) / (0.1 * ly)) ** 2)[:, None].expand(
        y.numel(), x.numel()).clone()
    v = torch.zeros_like(u)
    for xc, yc, r, p in torch.rand((12, 4), generator=g, dtype=torch.float64).tolist():
        r = (0.05 + 0.12 * r) * min(lx, ly)
        a = (2.0 * p - 1.0) * math.exp(0.5) / r
        gx = torch.exp(-(x - xc * lx) ** 2 / (2.0 * r * r))
        gy = torch.exp(-(y - yc * ly) ** 2 / (2.0 * r * r))
        u += torch.outer(a * (y - yc * ly) * gy, gx)
        v -= torch.outer(a * gy, (x - xc * lx) * gx)
    return u, v


def _scene(c, g, nx, ny, rays):
    """One scene's fields and rays as plain device tensors."""
    f = c["fields"]
    x, y = _axis(nx, c["dx"]), _axis(ny, c["dx"])
    lx, ly = float(x[-1]), float(y[-1])
    s = {"const": 50.0, "slope": (190.0, -150.0 / lx), "drift": (0.4, -0.2), "rays": rays}
    if f in ("shared", "separate", "depth"):
        s["bx"], s["by"], s["depth"] = x, y, _depth(g, x, y, c["bed"])
    if f in ("shared", "current"):
        s["cx"], s["cy"] = x, y
    elif f == "separate":
        q = c["ratio"]
        s["cx"] = torch.linspace(0.0, lx, max(8, int(nx / q)), dtype=torch.float64, device=DEV)
        s["cy"] = torch.linspace(0.0, ly, max(8, int(ny / q)), dtype=torch.float64, device=DEV)
    if "cx" in s:
        s["u"], s["v"] = _eddies(g, s["cx"], s["cy"])
    # launch points inside the grid, periods of wind sea and swell, all directions
    r = torch.rand((4, rays), generator=g, dtype=torch.float64).to(DEV)
    inner = 0.25 if c["entry"] in ("gradient", "iteration") and not c["rows"] else 0.02
    x0 = lx * (inner + (1.0 - 2.0 * inner) * r[0])
    y0 = ly * (inner + (1.0 - 2.0 * inner) * r[1])
    sigma = 2.0 * math.pi / (7.0 + 8.0 * r[2])
    if "depth" in s:
        h = s["depth"][(y0 / c["dx"]).round().long(), (x0 / c["dx"]).round().long()]
    elif f == "slope":
        h = s["slope"][0] + s["slope"][1] * x0
    else:
        h = torch.full_like(x0, s["const"])
    k = torch.maximum(sigma * sigma / G, sigma / torch.sqrt(G * h))
    for _ in range(12):
        th = torch.tanh(k * h)
        k = k - (G * k * th - sigma * sigma) / (G * th + G * k * h * (1.0 - th * th))
    a = 2.0 * math.pi * r[3]
    s["ic"] = [x0, y0, k * torch.cos(a), k * torch.sin(a)]
    return s


def _inputs(c, seed):
    g = torch.Generator().manual_seed(seed * 7919 + 17)
    if c["entry"] != "batch":
        return [_scene(c, g, c["nx"], c["ny"], c["rays"])]
    # grid sides and ray counts spread over a factor of about four and sixteen
    r = torch.rand((2, c["scenes"]), generator=torch.Generator().manual_seed(11),
                   dtype=torch.float64)
    w = torch.exp(r[1] * math.log(16.0))
    n = torch.clamp((w / w.sum() * c["rays"]).long(), min=1).tolist()
    side = (0.5 * torch.exp(r[0] * math.log(4.0))).tolist()
    return [_scene(c, g, max(16, int(c["nx"] * q)), max(16, int(c["ny"] * q)), m)
            for q, m in zip(side, n)]


def _targets(c, s, seed):
    """Where the rays of a gradient case should have gone, or row cotangents."""
    g = torch.Generator(device=DEV).manual_seed(seed + 5)
    n, nr = c["steps"] + 1, s["rays"]
    if c["rows"]:
        return [torch.randn((n, nr), generator=g, dtype=torch.float64, device=DEV)
                for _ in range(2)]
    d = 2.0 * torch.rand((nr, 2), generator=g, dtype=torch.float64, device=DEV) - 1.0
    return [torch.stack(s["ic"][:2], dim=1) + 2000.0 * d]


def _fields(s):
    if "depth" in s:
        b = Bathymetry.from_arrays(s["bx"].cpu().numpy(), s["by"].cpu().numpy(),
                                   s["depth"].cpu().numpy())
    elif s.get("plane"):
        b = Bathymetry.slope(h0=s["slope"][0], dhdx=s["slope"][1])
    else:
        b = Bathymetry.constant(s["const"])
    if "u" in s:
        cur = Current.from_arrays(s["cx"].cpu().numpy(), s["cy"].cpu().numpy(),
                                  s["u"].cpu().numpy(), s["v"].cpu().numpy())
    else:
        cur = Current.constant(*s["drift"])
    return b, cur


def prepare(case, seed):
    c = {**_DEFAULTS, **case}
    scenes = _inputs(c, seed)
    for s in scenes:
        s["plane"] = c["fields"] == "slope"
    T = (c["steps"] - 0.25) * c["dt"]      # a fraction of a step is rounded up to one
    st = {"case": c, "T": T}
    if c["entry"] == "batch":
        st["batch"] = Batch([dict(zip(("bathymetry", "current"), _fields(s)), t0=0.0, t_end=T,
                                  dt=c["dt"], **{k + "0": v for k, v in zip(STATE, s["ic"])})
                             for s in scenes], math=c["math"], solout=c["solout"])
        return st
    s = scenes[0]
    st["b"], st["c"] = _fields(s)
    if c["entry"] in ("single", "tracing"):
        st["ic"] = [v.cpu().numpy() for v in s["ic"]]
        return st
    st["ic"] = s["ic"]
    nr, n = c["rays"], c["steps"] + 1
    if c["entry"] == "device":
        f64 = dict(dtype=torch.float64, device=DEV)
        st["out"] = {"len": torch.empty(nr, dtype=torch.int32, device=DEV),
                     "end": torch.empty((nr, 4), **f64)}
        if c["rows"]:
            st["out"]["t"] = torch.empty(n, **f64)
            st["out"].update({k: torch.empty((n, nr), **f64) for k in STATE})
        return st
    st["to"] = _targets(c, s, seed)
    st["values"] = {k: s[k].reshape(-1) for k in ("depth", "u", "v") if k in s}
    if c["entry"] == "gradient":
        st["ic"] = [v.requires_grad_() for v in st["ic"]]
        st["values"] = {k: v.requires_grad_() for k, v in st["values"].items()}
    else:
        st["work"] = torch.empty(adjoint.workspace_bytes(nr, c["stride"]), dtype=torch.uint8,
                                 device=DEV)
    return st


# ---------------------------------------------------------------------------
# one pass

def run(state):
    c, T = state["case"], state["T"]
    kw = {"math": c["math"]}
    if c["entry"] == "batch":
        state["batch"].run()
        return state["batch"].results()
    b, cur, ic = state["b"], state["c"], state["ic"]
    if c["entry"] in ("single", "tracing"):
        if c["entry"] == "single":
            ds = core.single_ray(*[float(v[0]) for v in ic], T, c["dt"], b, cur, **kw)
        else:
            ds = core.ray_tracing(*ic, T, c["dt"], b, cur, **kw)
        return {k: ds[k].values for k in ("time",) + STATE}
    if c["entry"] == "device":
        return core.trace_many_device(b, cur, *ic, 0.0, T, c["dt"], trajectories=c["rows"],
                                      out=state["out"], precision=c["precision"],
                                      solout=c["solout"], **kw)
    val = state["values"]
    if c["entry"] == "gradient":
        out = adjoint.trace_differentiable(b, cur, *ic, 0.0, T, c["dt"], stride=c["stride"],
                                           trajectories=c["rows"], **val, **kw)
        wrt = ic + list(val.values())
        if c["rows"]:
            grads = torch.autograd.grad(out[2:4], wrt, state["to"])
        else:
            off = out[0][:, :2] - state["to"][0]
            loss = torch.where(torch.isnan(off), torch.zeros_like(off), off).square().sum()
            grads = torch.autograd.grad(loss, wrt)
        return {"end": out[0], "len": out[1], "grads": list(grads)}
    fwd = adjoint.trace_fp64(b, cur, *ic, 0.0, T, c["dt"], stride=c["stride"], **val, **kw)
    off = fwd["end"][:, :2] - state["to"][0]
    off = torch.where(torch.isnan(off).any(dim=1, keepdim=True), torch.zeros_like(off), off)
    g_end = torch.zeros_like(fwd["end"])
    g_end[:, :2] = 2.0 * off
    g = adjoint.adjoint(b, cur, fwd, 0.0, T, c["dt"], c["stride"], g_end=g_end,
                        want=tuple(val), work=state["work"], **val, **kw)
    return {"end": fwd["end"], "len": fwd["len"], "loss": off.square().sum(),
            "grads": [g[k] for k in val]}


def work(case):
    """Every ray takes every step (an upper bound where rays leave the grid);
    fields and launch states read once, rows, end states and gradients
    written once.  A backward pass repeats the forward's arithmetic and
    applies its transpose."""
    c = {**_DEFAULTS, **case}
    nr, n = c["rays"], c["steps"]
    cells = c["nx"] * c["ny"] * c["scenes"]
    grids = {"shared": 3.0, "separate": 1.0 + 2.0 / c["ratio"] ** 2, "depth": 1.0,
             "current": 2.0, "slope": 0.0}[c["fields"]] * cells * 8.0
    nbytes = grids + nr * (32 + 36)
    if c["rows"]:
        nbytes += 32.0 * nr * (n + 1) * (1.5 if c["entry"] == "gradient" else 1.0)
    flops = float(FLOP_PER_RAY_STEP) * nr * n
    if c["entry"] in ("gradient", "iteration"):
        nbytes += grids + 32.0 * nr
        flops *= 3.0
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------------------
# the same outputs in 64 bits from plain torch operations (f32 only where the
# reference's interpolation is defined in f32)

def _cell(p, axis, n):
    """Cell index along an axis and whether the point is on the grid."""
    q = ((p - axis[0]) / (axis[1] - axis[0]).abs()).detach()
    ok = (q >= 0) & (q <= n - 1)
    i = torch.clamp(torch.floor(torch.where(ok, q, torch.zeros_like(q))), 0, n - 2).long()
    return i, ok


def _corners(values, nx, i, j):
    a = nx * j + i
    return values[a], values[a + nx], values[a + nx + 1], values[a + 1]


def _bilinear(x, y, i, j, px, py, corners):
    """interpolator.rs:39-84 in the type of its arguments."""
    A, B, C, D = corners
    dtx, bty = x[i + 1] - x[i], y[j + 1] - y[j]
    det = -(dtx * bty)
    u, w = -(dtx / det) * (py - y[j]), -(bty / det) * (px - x[i])
    a10, a01 = B - A, D - A
    a11 = ((C - A) - a10) - a01
    return ((A + a10 * u) + a01 * w) + (a11 * u) * w


def _depth_at(s, px, py, f64):
    if s["plane"]:
        h0, sl = s["slope"]
        if f64:
            h0, sl = (float(torch.tensor(v, dtype=torch.float32)) for v in (h0, sl))
            return h0 + sl * px, sl, 0.0, ~torch.isnan(px + py)
        h0, sl = (torch.tensor(v, dtype=torch.float32, device=DEV) for v in (h0, sl))
        return (h0 + sl * px.float()).double(), sl.double(), 0.0, ~torch.isnan(px + py)
    if "depth" not in s:
        return torch.full_like(px, s["const"]), 0.0, 0.0, ~torch.isnan(px + py)
    x32, y32 = s["bx"].float(), s["by"].float()
    nx, ny = x32.numel(), y32.numel()
    x, y = (x32.double(), y32.double()) if f64 else (x32, y32)
    qx, qy = (px, py) if f64 else (px.float(), py.float())
    (i, oki), (j, okj) = _cell(qx, x, nx), _cell(qy, y, ny)
    c = _corners(s["depth_values"], nx, i, j)
    h = _bilinear(x, y, i, j, qx, qy, [v.to(x.dtype) for v in c])
    hx = (c[3] - c[0]) / (x32[1].double() - x32[0].double())
    hy = (c[1] - c[0]) / (y32[1].double() - y32[0].double())
    if not f64:
        hx, hy = hx.float().double(), hy.float().double()
    return h.double(), hx, hy, oki & okj


def _current_at(s, px, py, f64):
    if "u" not in s:
        return [s["drift"][0], 0.0, 0.0, s["drift"][1], 0.0, 0.0], True
    cx, cy = s["cx"], s["cy"]
    nx, ny = cx.numel(), cy.numel()
    (i, oki), (j, okj) = _cell(px, cx, nx), _cell(py, cy, ny)
    t = torch.float64 if f64 else torch.float32
    got = []
    for k in ("u_values", "v_values"):
        c = _corners(s[k], nx, i, j)
        got += [_bilinear(cx.to(t), cy.to(t), i, j, px.to(t), py.to(t),
                          [v.to(t) for v in c]).double(),
                (c[3] - c[0]) / (cx[1] - cx[0]), (c[1] - c[0]) / (cy[1] - cy[0])]
    return got, oki & okj


def _rhs(s, y, f64):
    px, py, kx, ky = y
    h, hx, hy, ok = _depth_at(s, px, py, f64)
    (u, ux, uy, v, vx, vy), okc = _current_at(s, px, py, f64)
    k = torch.sqrt(kx * kx + ky * ky)
    kh = k * h
    ok = ok & okc & (h > 0) & (k > 0)
    th, ch = torch.tanh(kh), torch.cosh(kh)
    cg = (G / 2.0) * ((th + kh / (ch * ch)) / torch.sqrt(k * G * th))
    cf = -0.5 * k / torch.sinh(kh) / ch * torch.sqrt(G * k * th)
    d = torch.stack([cg * kx / k + u, cg * ky / k + v, cf * hx - kx * ux - ky * vx,
                     cf * hy - kx * uy - ky * vy])
    return torch.where(ok, d, torch.full_like(d, math.nan))


def _step(s, y, dt, f64):
    k1 = _rhs(s, y, f64)
    k2 = _rhs(s, y + k1 * (dt / 2.0), f64)
    k3 = _rhs(s, y + k2 * (dt / 2.0), f64)
    k4 = _rhs(s, y + k3 * dt, f64)
    return y + (((k1 + k2 * 2.0) + k3 * 2.0) + k4) * (dt / 6.0), k1


def _exact_trace(c, s, f64, rows):
    y = torch.stack([v.detach() for v in s["ic"]])
    end, kept = y, [y]
    for i in range(c["steps"]):
        new, k1 = _step(s, y, c["dt"], f64)
        if c["solout"] == "next_deriv" and i > 0:
            stop = torch.isnan(k1).all(dim=0)
            end = torch.where(stop, end, new)
        else:
            end = torch.where(torch.isnan(y).all(dim=0), end, new)
        y = new
        if rows:
            kept.append(y)
    return end.T.contiguous(), kept


def _exact_gradients(c, s, states, seed):
    """Step by step backwards through the discrete map."""
    to = _targets(c, s, seed)
    names = [k for k in ("depth", "u", "v") if k in s]
    for k in names:
        s[k + "_values"].requires_grad_()
    par = [s[k + "_values"] for k in names]
    total = [torch.zeros_like(p) for p in par]
    lam = torch.zeros_like(states[0])
    if not c["rows"]:
        off = states[-1][:2] - to[0].T
        lam[:2] = torch.where(torch.isnan(off), torch.zeros_like(off), 2.0 * off)
    for i in range(c["steps"], -1, -1):
        if c["rows"]:
            ok = ~torch.isnan(states[i][:2])
            lam[:2] += torch.where(ok, torch.stack([t[i] for t in to]), torch.zeros_like(lam[:2]))
        if i == 0:
            break
        live = torch.nonzero(~torch.isnan(states[i]).any(dim=0))[:, 0]
        with torch.enable_grad():
            y = states[i - 1][:, live].requires_grad_()
            new, _ = _step(s, y, c["dt"], True)
            g = torch.autograd.grad(new, [y] + par, lam[:, live], allow_unused=True)
        lam = torch.zeros_like(lam)
        lam[:, live] = g[0]
        for t, v in zip(total, g[1:]):
            if v is not None:
                t += v
    return list(lam) + total


def exact(case, seed):
    c = {**_DEFAULTS, **case}
    if c["entry"] in ("batch", "iteration") or c["steps"] > 3000:
        return None
    s = _inputs(c, seed)[0]
    s["plane"] = c["fields"] == "slope"
    for k in ("depth", "u", "v"):
        if k in s:
            s[k + "_values"] = s[k].reshape(-1).clone()
    backward = c["entry"] == "gradient"
    f64 = backward or c["precision"] == "fp64"
    backward = backward and c["steps"] <= 700
    with torch.no_grad():
        end, kept = _exact_trace(c, s, f64, c["rows"] or backward)
    if c["entry"] == "gradient":
        n = len(s["ic"]) + sum(k in s for k in ("depth", "u", "v"))
        return {"end": end, "len": None,
                "grads": _exact_gradients(c, s, kept, seed) if backward else [None] * n}
    t = torch.arange(c["steps"] + 1, dtype=torch.float64, device=DEV) * c["dt"]
    if c["entry"] in ("single", "tracing"):
        rows = torch.stack(kept)                             # (n + 1, 4, rays)
        gone = torch.isnan(rows).all(dim=1)
        ln = torch.clamp((~gone).sum(dim=0) + 1, max=c["steps"] + 1)
        m = int(ln.max())
        i = torch.arange(m, device=DEV)[:, None]
        time = torch.where(i < ln[None, :], t[:m, None], torch.full_like(t[:m, None], math.nan))
        got = {"time": time, **{k: rows[:m, q] for q, k in enumerate(STATE)}}
        if c["entry"] == "single":
            got = {k: v[:, 0] for k, v in got.items()}
        return {k: v.contiguous() for k, v in got.items()}
    out = {"len": None, "end": end}
    if c["rows"]:
        rows = torch.stack(kept)
        out["t"] = t
        out.update({k: rows[:, q] for q, k in enumerate(STATE)})
    return out
