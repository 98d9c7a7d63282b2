"""The literal-math right-hand side over the whole range of wavenumbers and
depths, against the oracle's libm calls: kh from 1e-140 to 1e150 and beyond
both ends of exp, zero, negative, infinite and NaN depths, zero and NaN
wavenumbers.

NaNs fall where the oracle's do.  Finite values agree to 16 eps of the
column's scale, each side being within about 4 eps of the exact value; the
refraction factor, which carries exp(-2kh), has 2kh eps more on each side
from the rounding of k.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -52


@pytest.mark.parametrize("h0", [0.0, -3.0, 1e-30, 1e-3, 0.7, 50.0, 4000.0, 1e20, np.inf, np.nan])
def test_literal_range(oracle_mod, h0):
    import mantaray_amd as mr
    rng = np.random.default_rng(11)
    k = np.concatenate([10.0 ** rng.uniform(-140, 150, 400), 10.0 ** rng.uniform(-4, 1, 600)])
    th = rng.uniform(0.0, 2.0 * np.pi, k.size)
    s = np.zeros((k.size + 4, 4))
    s[:-4, 2], s[:-4, 3] = k * np.cos(th), k * np.sin(th)
    s[-3, 2], s[-2, 3], s[-1, 2:] = np.nan, 0.2, (-0.3, 0.0)
    hx, hy = 0.0125, -0.5                                # exact in f32
    got = mr.rhs(mr.Bathymetry.slope(h0, 0.0, 0.0, hx, hy), mr.Current.constant(0.0, 0.0), s,
                 math="literal")
    want = oracle_mod.system_many(oracle_mod.Bathymetry.slope(h0, 0.0, 0.0, hx, hy),
                                  oracle_mod.Current.constant(0.0, 0.0), s)[0]
    assert np.array_equal(np.isnan(got), np.isnan(want))
    fin = ~np.isnan(want).any(axis=1)
    if not fin.any():
        return
    kk = np.hypot(s[fin, 2], s[fin, 3])
    kh = np.minimum(kk * float(np.float32(h0)), 400.0)
    cg = np.hypot(want[fin, 0], want[fin, 1])
    dk = np.hypot(want[fin, 2], want[fin, 3])
    assert (np.abs(got[fin, :2] - want[fin, :2]) <= 16 * EPS * cg[:, None]).all()
    tol = (16 + 4 * kh) * EPS * dk + 1e-300
    assert (np.abs(got[fin, 2:] - want[fin, 2:]) <= tol[:, None]).all()
