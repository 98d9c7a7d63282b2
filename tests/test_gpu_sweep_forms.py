"""The reverse sweeps against each other where one could hide: the default
sweep past two workgroups a CU (one wave) against the two-wave kernel, the
flat-depth kernel after a forward in literal math, and gradients of some of a
pair's grids alone, whose other arrays the sums leave out.

All are sums of the same terms in other orders: equal to 1e-11 of each
gradient's scale, the bound of the other comparisons of sweeps.
"""
import itertools

import numpy as np
import pytest

from test_gpu_fp64_cells import _fields

pytestmark = pytest.mark.gpu

DT, T, STRIDE = 0.7, 6.5, 4


def _case(pair, n_rays, shared, math="fast"):
    import torch

    import mantaray_amd as mr
    from mantaray_amd import adjoint
    x, y, d, cx, cy, u, v = _fields(23, 14, "jittered", shared)
    rng = np.random.default_rng(n_rays)
    s = [torch.tensor(a, device="cuda:0") for a in
         (rng.uniform(x[2], x[-3], n_rays), rng.uniform(y[1], y[-2], n_rays),
          rng.uniform(-0.2, 0.2, n_rays), rng.uniform(-0.2, 0.2, n_rays))]
    b = (mr.Bathymetry.from_arrays(x.astype(np.float32), y.astype(np.float32), d)
         if pair != "current" else mr.Bathymetry.constant(30.0))
    c = mr.Current.from_arrays(cx, cy, u, v) if pair != "depth" else mr.Current.constant(0.2, -0.1)
    f = adjoint.trace_fp64(b, c, *s, 0.0, T, DT, stride=STRIDE, math=math)
    g = torch.tensor(rng.normal(size=(n_rays, 4)), device="cuda:0")

    def sweep(block, **kw):
        return adjoint.adjoint(b, c, f, 0.0, T, DT, STRIDE, g_end=g, block_size=block, math=math,
                               **kw)
    return sweep


def _agree(got, want):
    for k, w in want.items():
        assert (got[k] is None) == (w is None), k
        if w is not None:
            assert (got[k] - w).abs().max().item() <= 1e-11 * w.abs().max().item(), k


@pytest.mark.parametrize("pair", ["current", "depth", "both"])
@pytest.mark.parametrize("n_rays", [32_768, 32_769, 40_000])
def test_one_wave_default(pair, n_rays):
    sweep = _case(pair, n_rays, False)
    _agree(sweep(0), sweep(128))


@pytest.mark.parametrize("pair", ["current", "both"])
@pytest.mark.parametrize("n_rays", [16_385, 21_824, 21_825])
def test_between_one_and_two_workgroups_a_cu(pair, n_rays):
    """4/3 workgroups for each of 256 CUs are 341: 21,824 rays."""
    sweep = _case(pair, n_rays, False)
    got = sweep(0)
    _agree(got, sweep(64))
    _agree(got, sweep(128))
    _agree(got, sweep(256))


@pytest.mark.parametrize("n_rays", [1, 63, 65, 500])
def test_flat_depth_literal_forward(n_rays):
    sweep = _case("current", n_rays, False, "literal")
    want = sweep(128)
    _agree(sweep(64), want)
    _agree(sweep(256), want)


@pytest.mark.parametrize("shared", [True, False])
@pytest.mark.parametrize("block", [64, 128, 256])
def test_some_grids_alone(block, shared):
    sweep = _case("both", 300, shared)
    every = sweep(block)
    states = ("x0", "y0", "kx0", "ky0")
    for n in range(3):
        for grids in itertools.combinations(("depth", "u", "v"), n):
            got = sweep(block, want=states + grids)
            for k in ("depth", "u", "v"):
                assert (got[k] is not None) == (k in grids)
            _agree({k: got[k] for k in states + grids}, {k: every[k] for k in states + grids})
