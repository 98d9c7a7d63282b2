"""mr_field_upload builds all that a pair of fields without shared cells needs:
its first device trace then allocates nothing and can be captured in a HIP
graph.  And where the device has no memory for a field's own cell records,
traces run on the plain records, with the same results bitwise.
"""
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PAIRS = ("two grids", "depth only", "current only")


def _fields(pair, n=200):
    import mantaray_amd as mr
    x = 40.0 * np.arange(n)
    X, Y = np.meshgrid(x, x)
    b = (mr.Bathymetry.slope(40.0, 0.0, 0.0, -0.001, 0.002) if pair == "current only" else
         mr.Bathymetry.from_arrays(x, x, 20.0 + 5.0 * np.sin(X / 900.0) * np.cos(Y / 700.0)))
    c = (mr.Current.constant(0.3, -0.2) if pair == "depth only" else
         mr.Current.from_arrays(x * 1.01 - 9.0, x * 1.02 - 7.0, 0.4 * np.sin(Y / 800.0),
                                0.3 * np.cos(X / 600.0)))
    return b, c


def _rays(n):
    rng = np.random.default_rng(n)
    return [rng.uniform(500.0, 7000.0, n) for _ in range(2)] + [rng.uniform(-0.1, 0.1, n)
                                                                for _ in range(2)]


@pytest.mark.parametrize("pair", PAIRS)
def test_first_trace_captured_after_upload(pair):
    import torch

    import mantaray_amd as mr
    n, steps = 130, 40
    ic = [torch.tensor(v, device="cuda:0") for v in _rays(n)]
    want = mr.trace_many_device(*_fields(pair), *ic, 0.0, 0.7 * steps, 0.7)
    b, c = _fields(pair)
    b.upload(0)
    c.upload(0)
    out = {k: torch.zeros_like(v) for k, v in want.items()}
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        mr.trace_many_device(b, c, *ic, 0.0, 0.7 * steps, 0.7, out=out)
    for _ in range(3):
        for v in out.values():
            v.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for k, v in want.items():
            assert np.array_equal(out[k].cpu().numpy(), v.cpu().numpy(), equal_nan=True), k


@pytest.mark.parametrize("pair", PAIRS)
def test_first_trace_allocates_nothing_after_upload(pair):
    """On grids whose own records are tens of megabytes; and a second tile
    shape adds plain records, not another copy of the own ones."""
    import torch

    import mantaray_amd as mr
    n, cells = 64, 599 * 599
    ic = [torch.tensor(v, device="cuda:0") for v in _rays(n)]
    b, c = _fields(pair, 600)
    b.upload(0)
    c.upload(0)
    out = {k: torch.zeros(s, dtype=t, device="cuda:0") for k, s, t in
           (("len", n, torch.int32), ("end", (n, 4), torch.float64))}
    free = []
    for tile in (-1, -1, 0):
        mr.trace_many_device(b, c, *ic, 0.0, 7.0, 0.7, out=out, record_tile=tile)
        torch.cuda.synchronize()
        free.append(torch.cuda.mem_get_info()[0])
        if tile == -1 and len(free) == 1:
            # against the tables of other fields: the first trace took none
            b2, c2 = _fields(pair, 600)
            b2.upload(0)
            c2.upload(0)
            torch.cuda.synchronize()
            before = torch.cuda.mem_get_info()[0]
            mr.trace_many_device(b2, c2, *ic, 0.0, 7.0, 0.7, out=out)
            torch.cuda.synchronize()
            assert torch.cuda.mem_get_info()[0] >= before
            del b2, c2
            torch.cuda.synchronize()
            free[0] = torch.cuda.mem_get_info()[0]
    assert free[1] >= free[0]
    # plain records and raw values of a grid: 32 + 8 bytes a cell (depth), 64
    # + 8 + 16 (current), with 16 MiB for the axes and the allocations' grain
    grids = {"two grids": 40 + 88, "depth only": 40, "current only": 88}[pair]
    assert free[1] - free[2] <= 1.02 * grids * cells + (16 << 20)


SHIM = r"""
#include <cstddef>
extern "C" {
int (*real_malloc)(void **, size_t) = nullptr;
size_t limit = 0;                      // 0: none
int refused = 0;
int hipMalloc(void **p, size_t n)
{
    if (limit && n >= limit) {
        *p = nullptr;
        ++refused;
        return 2;                      // hipErrorOutOfMemory
    }
    return real_malloc(p, n);
}
}
"""

CHILD = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
import mantaray_amd as mr
from mantaray_amd import _capi as C
C.lib()
hip = [l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l][0]
real = ctypes.cast(ctypes.CDLL(hip).hipMalloc, ctypes.c_void_p).value
ctypes.c_void_p.in_dll(shim, "real_malloc").value = real
limit, refused = ctypes.c_size_t.in_dll(shim, "limit"), ctypes.c_int.in_dll(shim, "refused")
sys.path.insert(0, sys.argv[2])
from test_gpu_upload import PAIRS, _fields, _rays
N = 700
rays = _rays(300)
# below a gridded field's own records (64 and 128 bytes a cell), above its
# plain ones (32 and 64)
for pair in PAIRS:
    own = 699 * 699 * (64 if pair == "depth only" else 128)
    want = mr.trace_many(*_fields(pair, N), *rays, 0.0, 14.0, 0.7)
    assert refused.value == 0
    limit.value = own - 1000
    b, c = _fields(pair, N)
    before = 0
    for step in ("trace", "again", "uploaded"):
        got = mr.trace_many(b, c, *rays, 0.0, 14.0, 0.7)
        for k, v in want.items():
            assert np.array_equal(got[k], v, equal_nan=True), (pair, step, k)
        # asked for by a trace on new fields, not by one on the same fields
        # again, and by an upload
        asked, before = refused.value > before, refused.value
        assert asked == (step != "again"), step
        if step == "again":
            b.upload()
            c.upload()
    limit.value = 0
    b.upload()
    c.upload()
    limit.value = own - 1000
    got = mr.trace_many(b, c, *rays, 0.0, 14.0, 0.7)
    assert refused.value == before
    assert np.array_equal(got["x"], want["x"], equal_nan=True)
    limit.value = 0
    refused.value = 0
    print(pair, "ok", flush=True)
"""


def test_no_memory_for_own_records(tmp_path):
    """hipMalloc refused from the own records' size on, by a definition of it
    that stands before the runtime's in a child process."""
    src, so = tmp_path / "shim.cpp", str(tmp_path / "shim.so")
    src.write_text(SHIM)
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-o", so, str(src)], check=True)
    here = os.path.dirname(os.path.abspath(__file__))
    res = subprocess.run([sys.executable, "-u", "-c", CHILD, so, here], cwd=os.path.dirname(here),
                         capture_output=True, text=True, timeout=100)
    assert res.returncode == 0, res.stdout + res.stderr
    assert res.stdout.count("ok") == len(PAIRS)
