"""The one-wave sweep over a flat depth at stage points on the edge of the
data.  It forms a step's stage points again instead of reading them, so they
have to be the forward's own to the last bit: one unit in the last place
further, and a stage point that the forward evaluated on the grid's last node
lies off the grid, or in the next cell, whose values may be missing (NaN).

A uniform current over a constant depth leaves a ray's wavenumber alone, so
the four derivatives of a step are equal bitwise and its last stage point is
RN(dt dx/dt), exactly known.  The grid's last node (or the line to a cell
without data, one unit in the last place further) is put there, for rays of
many wavenumbers.  They start at x = 0 on the first node, so that no rounding
of the offsets from it hides that unit.  The gradient of the end's x with respect to the nodes' u
then sums to dt: the four products' weights, dt/6 (1 + 2 + 2 + 1), each spread
over corner weights that sum to one, and slope terms that cancel in the sum.
That is a few dozen rounded sums of terms no larger than about dt: 1e-12 of dt
is a wide bound for them, and a product left out changes the sum by a sixth.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT = 7.3
H = 20.0


def _rays(n=40):
    rng = np.random.default_rng(5)
    k, th = rng.uniform(0.02, 0.3, n), rng.uniform(-1.2, 1.2, n)
    return k * np.cos(th), k * np.sin(th)


@pytest.mark.parametrize("math", ["fast", "literal"])
@pytest.mark.parametrize("edge", ["last node", "cell without data"])
@pytest.mark.parametrize("block", [64, 128, 256])
def test_stage_points_on_the_edge(block, edge, math):
    import torch

    import mantaray_amd as mr
    from mantaray_amd import adjoint
    y = np.array([-900.0, 1100.0])
    b = mr.Bathymetry.constant(H)

    def uniform(x):
        u, v = np.full((2, x.size), 0.3), np.full((2, x.size), -0.1)
        return u, v

    kx, ky = _rays()
    wide = np.array([-1000.0, 0.0, 1000.0])
    c = mr.Current.from_arrays(wide, y, *uniform(wide))
    s = np.stack([np.zeros(kx.size), np.zeros(kx.size), kx, ky], axis=1)
    dx = mr.rhs(b, c, s, precision="fp64", math=math)[:, 0]
    assert (dx > 0.0).all()
    for i in range(kx.size):
        X = dx[i] * DT                              # the last stage point
        if edge == "last node":
            x = np.array([0.0, X])
            u, v = uniform(x)
        else:
            x = np.array([0.0, np.nextafter(X, np.inf), 1200.0])
            u, v = uniform(x)
            u[:, 2] = np.nan
        c = mr.Current.from_arrays(x, y, u, v)
        ic = [torch.tensor([q], dtype=torch.float64, device="cuda:0")
              for q in (0.0, 0.0, kx[i], ky[i])]
        f = adjoint.trace_fp64(b, c, *ic, 0.0, DT, DT, stride=1, math=math)
        assert bool(torch.isfinite(f["end"]).all()), i
        g = adjoint.adjoint(b, c, f, 0.0, DT, DT, 1, block_size=block, math=math,
                            g_end=torch.tensor([[1.0, 0.0, 0.0, 0.0]], dtype=torch.float64,
                                               device="cuda:0"))
        for k in ("x0", "y0", "kx0", "ky0"):
            assert bool(torch.isfinite(g[k]).all()), (i, k)
        assert abs(g["u"].sum().item() - DT) <= 1e-12 * DT, i
