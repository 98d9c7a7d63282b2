"""Host-array traces: the rows that come back through the pinned chunks equal
bitwise those the same launch leaves on the device, for sizes on both sides
of a chunk (4 MiB) and of a thread's share (1 MiB), for initial conditions
longer than a chunk, and from several threads at once; and the time rows of
ray_tracing against numpy, on the CPU.
"""
import threading

import numpy as np
import pytest

from mantaray_amd import _capi as C


@pytest.mark.parametrize("n_rows,n_rays", [(1, 1), (7, 3), (2, 700_001), (1201, 997)])
def test_time_rows(n_rows, n_rays):
    rng = np.random.default_rng(n_rows)
    t = np.cumsum(rng.uniform(0.1, 1.0, n_rows))
    ln = rng.integers(0, n_rows + 1, n_rays).astype(np.int32)
    out = np.full((n_rows, n_rays), 3.0)
    C.check(C.lib().mr_time_rows(n_rows, n_rays, t.ctypes.data, ln.ctypes.data, out.ctypes.data))
    want = np.where(np.arange(n_rows)[:, None] < ln[None, :], t[:, None], np.nan)
    assert np.array_equal(out, want, equal_nan=True)


def _states(n):
    rng = np.random.default_rng(n)
    s = [rng.uniform(0.0, 900.0, n) for _ in range(2)] + [rng.uniform(-0.2, 0.2, n) for _ in range(2)]
    s[2][: min(n, 3)] = 0.0
    s[3][: min(n, 3)] = 0.0                              # k = 0: these rays end at once
    return s


@pytest.mark.gpu
@pytest.mark.parametrize("n_rays,steps", [(1, 5), (1, 0), (129, 250), (131, 249), (1000, 130),
                                          (150_001, 2), (3001, 400)])
@pytest.mark.parametrize("trajectories", [True, False])
def test_host_rows_equal_device_rows(n_rays, steps, trajectories):
    import torch

    import mantaray_amd as mr
    b, c = mr.Bathymetry.slope(40.0, 0.0, 0.0, -0.01, 0.003), mr.Current.constant(0.2, -0.1)
    s = _states(n_rays)
    T = 0.7 * steps
    want = mr.trace_many_device(b, c, *[torch.tensor(v, device="cuda:0") for v in s], 0.0, T, 0.7,
                                trajectories=trajectories)
    want = {k: None if v is None else v.cpu().numpy() for k, v in want.items()}
    got = [None] * 3

    def call(i):
        got[i] = mr.trace_many(b, c, *s, 0.0, T, 0.7, trajectories=trajectories)

    call(0)
    threads = [threading.Thread(target=call, args=(i,)) for i in (1, 2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g in got:
        for k, v in want.items():
            assert (g[k] is None) == (v is None), k
            if v is not None:
                assert np.array_equal(g[k], v, equal_nan=True), k


@pytest.mark.gpu
def test_no_rays():
    import mantaray_amd as mr
    e = np.zeros(0)
    r = mr.trace_many(mr.Bathymetry.constant(10.0), mr.Current.constant(), e, e, e, e, 0.0, 3.0, 1.0)
    assert r["x"].shape == (4, 0) and r["len"].size == 0
    assert np.array_equal(r["t"], [0.0, 1.0, 2.0, 3.0])
