"""Traces by what their axes are: the route a pair of fields takes (its own
cell records, or the plain ones where too many targets lie outside the cells'
fast regions), both against the oracle, and points within two units in the
last place of the cell lines.

Row counts and NaN patterns are the oracle's, positions within 1e-6 m and
wavenumbers within 1e-8 of their scale (the tolerances of the other trace
tests); after one step of 0.01 s, 1e-12 of the scale: the derivatives are the
oracle's to some 1e-14, and those of a neighbouring cell differ by their own
size, 1e-4 of the scale and more in a step.
"""
import os
import subprocess
import sys

import numpy as np
import pytest

from test_gpu_plain_records import SHIM

pytestmark = pytest.mark.gpu

# (offset, spacing, nodes) of square grids, and whether depth alone, the
# current alone and both run on own records: the share of targets outside is
# about 2, 3 and 5 times the f32 spacing's share of a cell
AXES = {
    "near": (0.0, 40.0, 60, True, True, True),
    "1/1600 of a cell": (5.0e5, 50.0, 60, True, True, False),
    "1/160 of a cell": (2.0e6, 20.0, 60, False, False, False),
    "first spacing off": (5.0e5, 33.333, 60, False, False, False),
}
PAIRS = ("depth only", "current only", "two grids")


def _made(M, mr, pair, off, sp, n, seed=1):
    rng = np.random.default_rng(seed)
    x = off + sp * np.arange(n)
    X, Y = np.meshgrid(x - off, x - off)
    d = 20.0 + 6.0 * np.sin(X / (7.0 * sp)) * np.cos(Y / (9.0 * sp)) + rng.normal(0.0, 0.5, X.shape)
    U = 0.5 * np.sin(Y / (8.0 * sp)) + rng.normal(0.0, 0.05, X.shape)
    V = 0.4 * np.cos(X / (6.0 * sp)) + rng.normal(0.0, 0.05, X.shape)
    grid = M.Bathymetry.from_arrays if M is mr else M.Bathymetry.grid
    cur = M.Current.from_arrays if M is mr else M.Current.grid
    b = (M.Bathymetry.constant(12.5) if pair == "current only" else
         grid(x.astype(np.float32), x.astype(np.float32), d))
    c = (M.Current.constant(0.3, -0.2) if pair == "depth only" else
         cur(x - 0.25 * sp, x - 0.5 * sp, U, V))
    return b, c


def _rays(off, sp, n, nr, seed=2):
    rng = np.random.default_rng(seed)
    return [rng.uniform(off - sp, off + sp * n, nr) for _ in range(2)] + [
        rng.uniform(-0.15, 0.15, nr) for _ in range(2)]


CHILD = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import mantaray_amd as mr
from mantaray_amd import _capi as C
C.lib()
hip = ctypes.CDLL([l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l][0])
for name, fn in (("real_malloc", hip.hipMalloc), ("real_launch", hip.hipLaunchKernel)):
    ctypes.c_void_p.in_dll(shim, name).value = ctypes.cast(fn, ctypes.c_void_p).value
last = (ctypes.c_char * 512).in_dll(shim, "last")
sys.path.insert(0, sys.argv[2])
from test_gpu_axis_routes import AXES, PAIRS, _made, _rays
for name, (off, sp, n, *own) in AXES.items():
    for pair, o in zip(PAIRS, own):
        b, c = _made(mr, mr, pair, off, sp, n)
        mr.trace_many(b, c, *_rays(off, sp, n, 70), 0.0, 3.0, 0.7)
        rec = last.value.decode().split("trace_kernel")[1].split("E")[4]
        print(name, pair, "own" if rec == "Li2" else "plain" if rec == "Li0" else rec,
              "expected", "own" if o else "plain", flush=True)
"""


def test_route(tmp_path):
    src, so = tmp_path / "shim.cpp", str(tmp_path / "shim.so")
    src.write_text(SHIM)
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-o", so, str(src), "-ldl"], check=True)
    here = os.path.dirname(os.path.abspath(__file__))
    res = subprocess.run([sys.executable, "-u", "-c", CHILD, so, here], cwd=os.path.dirname(here),
                         capture_output=True, text=True, timeout=100)
    assert res.returncode == 0, res.stdout + res.stderr
    rows = [ln.split() for ln in res.stdout.splitlines() if " expected " in ln]
    assert len(rows) == len(AXES) * len(PAIRS)
    assert all(r[-3] == r[-1] for r in rows), res.stdout


@pytest.mark.parametrize("pair", PAIRS)
@pytest.mark.parametrize("axes", AXES)
@pytest.mark.parametrize("dt", [0.5, 1.3])
def test_against_oracle(oracle_mod, axes, pair, dt):
    import mantaray_amd as mr
    off, sp, n, *_ = AXES[axes]
    s = _rays(off, sp, n, 200)
    args = (*s, 0.0, 24.75 * dt, dt)
    ref = oracle_mod.trace_many(*_made(oracle_mod, mr, pair, off, sp, n), *args)
    got = mr.trace_many(*_made(mr, mr, pair, off, sp, n), *args)
    assert np.array_equal(got["len"], ref["len"])
    for k in ("x", "y", "kx", "ky"):
        assert np.array_equal(np.isnan(got[k]), np.isnan(ref[k])), k
    assert max(np.nanmax(np.abs(got[k] - ref[k])) for k in ("x", "y")) <= 1e-6
    scale = np.nanmax(np.abs(ref["kx"])) + np.nanmax(np.abs(ref["ky"]))
    assert max(np.nanmax(np.abs(got[k] - ref[k])) for k in ("kx", "ky")) <= 1e-8 * scale


@pytest.mark.parametrize("n_rays", [65_536, 65_537, 70_001])
def test_more_waves_than_simds_on_own_records(n_rays):
    """On both sides of the ray count at which waves share SIMDs, single and
    in a batch of two scenes: the end states of a few rays, bitwise."""
    import torch

    import mantaray_amd as mr
    from mantaray_amd.batch import Batch
    off, sp, n, *_ = AXES["near"]
    b, c = _made(mr, mr, "two grids", off, sp, n)
    s = _rays(off, sp, n, 300)
    few = mr.trace_many(b, c, *s, 0.0, 11.0, 0.7, trajectories=False)
    i = np.arange(n_rays) % 300
    ic = [torch.tensor(np.ascontiguousarray(v[i]), device="cuda:0") for v in s]
    many = mr.trace_many_device(b, c, *ic, 0.0, 11.0, 0.7, trajectories=False)
    assert np.array_equal(many["len"].cpu().numpy(), few["len"][i])
    assert np.array_equal(many["end"].cpu().numpy(), few["end"][i], equal_nan=True)
    batch = Batch([{"bathymetry": b, "current": c, "t0": 0.0, "t_end": 11.0, "dt": 0.7,
                    **{k: v[p] for k, v in zip(("x0", "y0", "kx0", "ky0"), ic)}}
                   for p in (slice(0, n_rays // 2), slice(n_rays // 2, None))])
    batch.run()
    end = torch.cat([o["end"] for o in batch.results()]).cpu().numpy()
    assert np.array_equal(end, few["end"][i], equal_nan=True)
    batch.close()


@pytest.mark.parametrize("precision", ["reference", "fp64"])
@pytest.mark.parametrize("grids", ["depth", "current", "shared", "apart"])
@pytest.mark.parametrize("a0,sp,n", [(0.0, 40.0, 12), (-7.0, 7.0, 3), (1.0e5, 128.0, 9),
                                     (-1000.0, 0.1, 41), (1.0e7, 3.3, 17), (2.0, -0.7, 12)])
def test_cell_lines(oracle_mod, a0, sp, n, grids, precision):
    import mantaray_amd as mr
    x = (a0 + sp * np.arange(n)).astype(np.float32).astype(np.float64)
    y = np.array([0.0, 10.0, 20.0])
    cy = y if grids != "apart" else np.append(y, 31.0)
    rng = np.random.default_rng(n)
    depth = rng.uniform(8.0, 30.0, (3, n))
    U, V = rng.uniform(-1.0, 1.0, (2, cy.size, n))
    px = []
    for f in (np.float32, np.float64):
        for to in (-np.inf, np.inf):
            q = x.astype(f)
            for _ in range(3):
                px.append(q.astype(np.float64))
                q = np.nextafter(q, f(to))
    px = np.concatenate(px)
    # away from the lines too, where the cells' own regions serve
    px = np.append(px, rng.uniform(x.min(), x.max(), 40))
    s = [px, np.full(px.size, 6.5), np.full(px.size, 0.07), np.full(px.size, -0.03)]
    made = []
    for M in (mr, oracle_mod):
        grid = M.Bathymetry.from_arrays if M is mr else M.Bathymetry.grid
        cur = M.Current.from_arrays if M is mr else M.Current.grid
        b = (M.Bathymetry.constant(12.5) if grids == "current" else
             grid(x.astype(np.float32), y.astype(np.float32), depth))
        c = M.Current.constant(0.3, -0.2) if grids == "depth" else cur(x, cy, U, V)
        made.append((b, c))
    prec = oracle_mod.PREC_FP64_INTERP if precision == "fp64" else 0
    ref = oracle_mod.trace_many(*made[1], *s, 0.0, 0.01, 0.01, prec=prec)
    got = mr.trace_many(*made[0], *s, 0.0, 0.01, 0.01, precision=precision)
    assert np.array_equal(got["len"], ref["len"])
    for k in ("x", "y", "kx", "ky"):
        assert np.array_equal(np.isnan(got[k]), np.isnan(ref[k])), k
    assert np.isfinite(ref["kx"][1]).any()
    scale = np.nanmax(np.abs(ref["kx"])) + np.nanmax(np.abs(ref["ky"]))
    assert max(np.nanmax(np.abs(got[k] - ref[k])) for k in ("kx", "ky")) <= 1e-12 * scale


@pytest.mark.parametrize("order", [("near", "1/160 of a cell"), ("1/160 of a cell", "near")])
@pytest.mark.parametrize("pair", PAIRS)
def test_batch_over_both_routes(pair, order):
    """A batch runs on one kind of records: on the plain ones when any of its
    scenes does, in whatever order they come.  The end states are those of a
    trace of each scene, bitwise."""
    import torch

    import mantaray_amd as mr
    from mantaray_amd.batch import Batch
    scenes, want = [], []
    for name in order:
        off, sp, n, *_ = AXES[name]
        b, c = _made(mr, mr, pair, off, sp, n)
        s = _rays(off, sp, n, 150)
        want.append(mr.trace_many(b, c, *s, 0.0, 11.0, 0.7, trajectories=False))
        scenes.append({"bathymetry": b, "current": c, "t0": 0.0, "t_end": 11.0, "dt": 0.7,
                       **dict(zip(("x0", "y0", "kx0", "ky0"), s))})
    batch = Batch(scenes)
    batch.run()
    torch.cuda.synchronize()
    for got, w in zip(batch.results(), want):
        assert np.array_equal(got["len"].cpu().numpy(), w["len"])
        assert np.array_equal(got["end"].cpu().numpy(), w["end"], equal_nan=True)
    batch.close()


@pytest.mark.parametrize("pair", PAIRS)
@pytest.mark.parametrize("axes", ["near", "1/160 of a cell"])
def test_data_shorter_than_the_grid(oracle_mod, axes, pair):
    """Value arrays that end two rows and a few nodes early: the cells with a
    corner past them err, on either route."""
    import mantaray_amd as mr
    off, sp, n, *_ = AXES[axes]
    made = []
    for M in (mr, oracle_mod):
        rng = np.random.default_rng(4)
        x = off + sp * np.arange(n)
        d, U, V = rng.uniform(9.0, 30.0, n * n), *rng.uniform(-0.6, 0.6, (2, n * n))
        grid = M.Bathymetry.from_arrays if M is mr else M.Bathymetry.grid
        cur = M.Current.from_arrays if M is mr else M.Current.grid
        made.append((M.Bathymetry.constant(12.5) if pair == "current only" else
                     grid(x.astype(np.float32), x.astype(np.float32), d[:-2 * n - 3]),
                     M.Current.constant(0.3, -0.2) if pair == "depth only" else
                     cur(x - 0.25 * sp, x - 0.5 * sp, U[:-n - 7], V[:-2 * n - 1])))
    args = (*_rays(off, sp, n, 300, 7), 0.0, 18.75, 0.75)
    ref = oracle_mod.trace_many(*made[1], *args)
    got = mr.trace_many(*made[0], *args)
    assert np.array_equal(got["len"], ref["len"])
    for k in ("x", "y", "kx", "ky"):
        assert np.array_equal(np.isnan(got[k]), np.isnan(ref[k])), k
    assert max(np.nanmax(np.abs(got[k] - ref[k])) for k in ("x", "y")) <= 1e-6
    scale = np.nanmax(np.abs(ref["kx"])) + np.nanmax(np.abs(ref["ky"]))
    assert max(np.nanmax(np.abs(got[k] - ref[k])) for k in ("kx", "ky")) <= 1e-8 * scale
