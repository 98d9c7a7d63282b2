"""Traces on each gridded field's own cell records, and on the plain records
that grids too large for them use, against the oracle.

The own records serve every pair that does not share cells: two grids, a
gridded depth under a constant current, and a gridded current over an
analytic depth.  Grids from a single cell up, with jittered and descending
axes among them; states on nodes, on cell lines, off the grid and NaN; a
step that is a power of two (one rounding per stage state) and one that is
not; both math modes and both solout readings.  Row counts and NaN patterns
are identical, positions within 1e-6 m, wavenumbers within 1e-8 of their
scale (the tolerances of the other trace tests), and a batch of two scenes
gives the traces' end states bitwise.
"""
import numpy as np
import pytest

from _helpers import random_states

pytestmark = pytest.mark.gpu

PAIRS = ("two grids", "depth only", "current only", "slope", "array")


@pytest.fixture(scope="module")
def mr():
    import mantaray_amd
    from mantaray_amd import _capi
    _capi.lib()
    return mantaray_amd


def _axes(rng, n, form):
    a = 40.0 * np.arange(n) + 3.0
    if form == "jittered":
        a[1:] += rng.uniform(-8.0, 8.0, n - 1)
    elif form == "descending":
        a = a[::-1].copy()
    return a.astype(np.float32).astype(np.float64)


def _fields(mr, oracle_mod, pair, nx, ny, form):
    rng = np.random.default_rng(nx * 1000 + ny)
    x, y = _axes(rng, nx, form), _axes(rng, ny, "uniform")
    X, Y = np.meshgrid(x, y)
    depth = 14.0 + 8.0 * np.sin(X / 90.0) * np.cos(Y / 70.0) + rng.normal(0.0, 1.0, X.shape)
    # the current's own grid covers the depth's, with other cells
    cx = np.linspace(x.min() - 11.0, x.max() + 7.0, max(2, nx - 1))
    cy = np.linspace(y.min() - 5.0, y.max() + 13.0, max(2, ny // 2 + 1))
    U = 0.6 * np.sin(cy / 80.0)[:, None] + rng.normal(0.0, 0.1, (cy.size, cx.size))
    V = 0.5 * np.cos(cx / 60.0)[None, :] + rng.normal(0.0, 0.1, (cy.size, cx.size))
    made = []
    for M in (mr, oracle_mod):
        grid = M.Bathymetry.from_arrays if M is mr else M.Bathymetry.grid
        cur = M.Current.from_arrays if M is mr else M.Current.grid
        b = {"two grids": lambda: grid(x.astype(np.float32), y.astype(np.float32), depth),
             "depth only": lambda: grid(x.astype(np.float32), y.astype(np.float32), depth),
             "current only": lambda: M.Bathymetry.constant(12.5),
             "slope": lambda: M.Bathymetry.slope(20.0, 0.0, 0.0, -0.01, 0.004),
             "array": lambda: M.Bathymetry.array(
                 (6.0 + (np.arange(700 * 700) % 13)).reshape(700, 700).astype(np.float32))}[pair]()
        c = M.Current.constant(0.3, -0.2) if pair == "depth only" else cur(cx, cy, U, V)
        made.append((b, c))
    cfg = {"bathy": {"x": np.sort(x), "y": y}}
    return made, random_states(nx + ny, cfg, 256) if min(nx, ny) > 3 else _few_states(x, y)


def _few_states(x, y):
    rng = np.random.default_rng(4)
    s = np.stack([rng.uniform(x.min() - 9.0, x.max() + 9.0, 96),
                  rng.uniform(y.min() - 9.0, y.max() + 9.0, 96),
                  rng.uniform(-0.1, 0.1, 96), rng.uniform(-0.1, 0.1, 96)], axis=1)
    s[:8, 0] = rng.choice(x, 8)
    s[4:12, 1] = rng.choice(y, 8)
    return s


@pytest.mark.parametrize("pair", PAIRS)
@pytest.mark.parametrize("nx,ny,form,dt", [(2, 2, "uniform", 1.0), (3, 17, "uniform", 0.7),
                                           (34, 9, "jittered", 0.5), (13, 21, "descending", 1.3)])
def test_own_records(mr, oracle_mod, pair, nx, ny, form, dt):
    ((b, c), (ob, oc)), s = _fields(mr, oracle_mod, pair, nx, ny, form)
    steps = 25
    T = (steps - 0.25) * dt
    for math in ("fast", "literal"):
        for solout in ("state", "next_deriv"):
            osol = oracle_mod.SOLOUT_STATE if solout == "state" else oracle_mod.SOLOUT_NEXT_DERIV
            ref = oracle_mod.trace_many(ob, oc, *s.T.copy(), 0.0, T, dt, solout=osol)
            got = mr.trace_many(b, c, *s.T, 0.0, T, dt, math=math, solout=solout)
            assert np.array_equal(got["len"], ref["len"])
            for k in ("x", "y", "kx", "ky"):
                assert np.array_equal(np.isnan(got[k]), np.isnan(ref[k])), k
            assert max(np.nanmax(np.abs(got[k] - ref[k])) for k in ("x", "y")) <= 1e-6
            scale = np.nanmax(np.abs(ref["kx"])) + np.nanmax(np.abs(ref["ky"]))
            assert max(np.nanmax(np.abs(got[k] - ref[k])) for k in ("kx", "ky")) <= 1e-8 * scale
    from mantaray_amd.batch import Batch
    import torch
    half = s.shape[0] // 2
    scenes = [{"bathymetry": b, "current": c, "t0": 0.0, "t_end": T, "dt": dt,
               **{k: p[:, q] for q, k in enumerate(("x0", "y0", "kx0", "ky0"))}}
              for p in (s[:half], s[half:])]
    batch = Batch(scenes)
    batch.run()
    torch.cuda.synchronize()
    ref = mr.trace_many(b, c, *s.T, 0.0, T, dt, trajectories=False)
    out = batch.results()
    assert np.array_equal(np.concatenate([o["len"].cpu().numpy() for o in out]), ref["len"])
    assert np.array_equal(np.concatenate([o["end"].cpu().numpy() for o in out]), ref["end"],
                          equal_nan=True)
    batch.close()


@pytest.mark.parametrize("nx", [2 ** 23 + 3, 2 ** 21])
def test_grid_past_the_record_limit(mr, oracle_mod, nx):
    """A current of 4 x 8.4 million cells: its 128-byte records pass 4 GiB,
    so the trace runs on the plain records; a quarter of it does not."""
    ny = 5
    cx, cy = 4.0 * np.arange(nx), 30.0 * np.arange(ny)
    u = np.broadcast_to(0.4 * np.sin(cx / 500.0)[None, :], (ny, nx)).ravel()
    v = np.repeat(0.1 * np.cos(cy / 20.0), nx)
    rng = np.random.default_rng(3)
    s = np.stack([rng.uniform(0.0, cx[-1], 128), rng.uniform(20.0, 100.0, 128),
                  rng.uniform(-0.1, 0.1, 128), rng.uniform(-0.02, 0.02, 128)], axis=1)
    # rays near the last cells, where the records' byte offsets are largest
    s[:32, 0] = cx[-1] - rng.uniform(0.0, 60.0, 32)
    args = (*s.T.copy(), 0.0, 20.0, 1.0)
    ref = oracle_mod.trace_many(oracle_mod.Bathymetry.constant(15.0),
                                oracle_mod.Current.grid(cx, cy, u, v), *args)
    got = mr.trace_many(mr.Bathymetry.constant(15.0), mr.Current.from_arrays(cx, cy, u, v), *args,
                        record_tile=0)
    assert np.array_equal(got["len"], ref["len"])
    for k, tol in (("x", 1e-6), ("y", 1e-6), ("kx", 1e-9), ("ky", 1e-9)):
        assert np.array_equal(np.isnan(got[k]), np.isnan(ref[k]))
        assert np.nanmax(np.abs(got[k] - ref[k])) <= tol


@pytest.mark.parametrize("n_rays", [65_536, 65_537, 70_001])
def test_more_waves_than_simds(mr, oracle_mod, n_rays):
    """Two gridded fields on grids of their own, on both sides of the ray
    count at which waves share SIMDs (256 CUs x 256 lanes): the same rays as
    in a launch of a few give the same end states bitwise, in single traces
    and in batches of two scenes."""
    import torch

    from mantaray_amd.batch import Batch
    ((b, c), _), s = _fields(mr, oracle_mod, "two grids", 34, 9, "jittered")
    few = mr.trace_many(b, c, *s.T, 0.0, 11.0, 0.7, trajectories=False)
    i = np.arange(n_rays) % s.shape[0]
    ic = [torch.tensor(np.ascontiguousarray(s[i, q]), device="cuda:0") for q in range(4)]
    many = mr.trace_many_device(b, c, *ic, 0.0, 11.0, 0.7, trajectories=False)
    assert np.array_equal(many["len"].cpu().numpy(), few["len"][i])
    assert np.array_equal(many["end"].cpu().numpy(), few["end"][i], equal_nan=True)
    half = n_rays // 2
    batch = Batch([{"bathymetry": b, "current": c, "t0": 0.0, "t_end": 11.0, "dt": 0.7,
                    **{k: v[p] for k, v in zip(("x0", "y0", "kx0", "ky0"), ic)}}
                   for p in (slice(0, half), slice(half, None))])
    batch.run()
    end = torch.cat([o["end"] for o in batch.results()]).cpu().numpy()
    assert np.array_equal(end, few["end"][i], equal_nan=True)
    batch.close()


@pytest.mark.parametrize("a0,sp,n", [(-1000.0, 0.1, 41), (-7.0, 7.0, 3), (1.0e7, 3.3, 17),
                                     (3.0e-30, 7.0e-31, 9), (2.0, -0.7, 12), (-2.0e30, 1.7e29, 30)])
def test_cell_lines_of_awkward_axes(mr, oracle_mod, a0, sp, n):
    """Points within two units in the last place of every cell line, in f32
    and f64, on axes that cross zero, lie far from it, descend, or have
    extreme spacings: the cell each falls in, seen in the cell's slopes, is
    the oracle's.  A neighbouring cell's slope differs by order one; the
    tolerance is that of the right-hand-side tests."""
    x = a0 + sp * np.arange(n)
    x = x.astype(np.float32).astype(np.float64)
    y = np.array([0.0, 10.0, 20.0])
    rng = np.random.default_rng(n)
    depth = rng.uniform(8.0, 30.0, (3, n))
    U, V = rng.uniform(-1.0, 1.0, (2, 3, n))
    px = []
    for f in (np.float32, np.float64):
        for to in (-np.inf, np.inf):
            q = x.astype(f)
            for _ in range(3):
                px.append(q.astype(np.float64))
                q = np.nextafter(q, f(to))
    px = np.concatenate(px)
    s = np.stack([px, np.full(px.size, 6.5), np.full(px.size, 0.07),
                  np.full(px.size, -0.03)], axis=1)
    y32 = y.astype(np.float32)
    for grid in ("depth", "current"):
        if grid == "depth":
            b, ob = (g(x.astype(np.float32), y32, depth)
                     for g in (mr.Bathymetry.from_arrays, oracle_mod.Bathymetry.grid))
            c, oc = mr.Current.constant(0.3, -0.2), oracle_mod.Current.constant(0.3, -0.2)
        else:
            b, ob = mr.Bathymetry.constant(12.5), oracle_mod.Bathymetry.constant(12.5)
            c, oc = (g(x, y, U, V) for g in (mr.Current.from_arrays, oracle_mod.Current.grid))
        ds = mr.rhs(b, c, s, math="literal")
        ref, _ = oracle_mod.system_many(ob, oc, s)
        assert np.array_equal(np.isnan(ds), np.isnan(ref)), grid
        assert np.isfinite(ref).any(), grid
        ok = np.isfinite(ref)
        scale = np.max(np.abs(np.where(ok, ref, 0.0)), axis=0)
        assert np.array_equal(ds[~ok & ~np.isnan(ref)], ref[~ok & ~np.isnan(ref)]), grid
        assert np.max(np.abs(ds - ref)[ok] / np.broadcast_to(scale, ds.shape)[ok]) <= 1e-12, grid
