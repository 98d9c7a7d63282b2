"""Points a subnormal number below the first node: their fractional index,
(p - a0)/spacing, underflows to -0, which is not below zero, so they are on
the grid (cartesian_current.rs:244-262).  The right-hand side and the first
step of a trace put them there on every route, as the oracle does.  The
derivatives' tolerance is that of the right-hand-side tests; after a step of
0.01 s it is one unit in the last place of the state more.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TINY = 5e-324


@pytest.mark.parametrize("precision", ["reference", "fp64"])
@pytest.mark.parametrize("grids", ["depth", "current", "shared", "apart"])
@pytest.mark.parametrize("sp", [40.0, 3.0, 0.3])
def test_first_node(oracle_mod, grids, sp, precision):
    import mantaray_amd as mr
    x, y = sp * np.arange(6), np.array([0.0, 10.0, 20.0])
    cy = y if grids != "apart" else np.append(y, 31.0)
    rng = np.random.default_rng(6)
    depth = rng.uniform(8.0, 30.0, (3, x.size))
    U, V = rng.uniform(-1.0, 1.0, (2, cy.size, x.size))
    px = np.array([m * TINY for m in (-41, -40, -21, -20, -19, -3, -2, -1, 0, 1, 2)]
                  + [-0.0, -1e-300, -1e-45, -1e-46, -1e-44, -1e-20])
    s = np.stack([px, np.full(px.size, 6.5), np.full(px.size, 0.07), np.full(px.size, -0.03)], axis=1)
    made = []
    for M in (mr, oracle_mod):
        grid = M.Bathymetry.from_arrays if M is mr else M.Bathymetry.grid
        cur = M.Current.from_arrays if M is mr else M.Current.grid
        b = (M.Bathymetry.constant(12.5) if grids == "current" else
             grid(x.astype(np.float32), y.astype(np.float32), depth))
        c = M.Current.constant(0.3, -0.2) if grids == "depth" else cur(x, cy, U, V)
        made.append((b, c))
    prec = oracle_mod.PREC_FP64_INTERP if precision == "fp64" else oracle_mod.PREC_REFERENCE
    ref, _ = oracle_mod.system_many(*made[1], s, prec=prec)
    ds = mr.rhs(*made[0], s, precision=precision)
    assert np.array_equal(np.isnan(ds), np.isnan(ref))
    if sp > 2.0:                                         # (else -TINY/sp does not underflow)
        assert np.isfinite(ref[7]).all()
    scale = np.nanmax(np.abs(ref), axis=0)
    assert np.nanmax(np.abs(ds - ref) / scale) <= 1e-12
    ref = oracle_mod.trace_many(*made[1], *s.T.copy(), 0.0, 0.01, 0.01, prec=prec)
    got = mr.trace_many(*made[0], *s.T, 0.0, 0.01, 0.01, precision=precision)
    assert np.array_equal(got["len"], ref["len"])
    for k in ("x", "y", "kx", "ky"):
        assert np.array_equal(np.isnan(got[k]), np.isnan(ref[k])), k
        assert np.nanmax(np.abs(got[k] - ref[k])) <= 1e-12 * np.nanmax(np.abs(ref[k])), k
