"""The buffers that host-memory traces keep between calls, seen through
definitions of the allocating HIP calls that stand before the runtime's in a
child process: calls on file paths, which open and free their fields each
time, make no stream and no pinned chunk again; a chunk is no larger than its
call needs; a call does with the workers it has when pinned memory is refused,
and gives idle buffers back when device memory is; and all of it can be
released."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

SHIM = r"""
#include <cstddef>
extern "C" {
int (*real_malloc)(void **, size_t) = nullptr;
int (*real_host)(void **, size_t, unsigned) = nullptr;
int (*real_host_free)(void *) = nullptr;
int (*real_stream)(void **, unsigned) = nullptr;
int (*real_destroy)(void *) = nullptr;
int streams = 0, destroyed = 0, pins = 0, unpinned = 0, refused = 0;
int pins_left = -1;                    // pinned allocations granted; -1: all
int refuse_once = 0;                   // device allocations refused
size_t pinned = 0, largest = 0;
int hipMalloc(void **p, size_t n)
{
    if (refuse_once) {
        --refuse_once;
        ++refused;
        *p = nullptr;
        return 2;                      // hipErrorOutOfMemory
    }
    return real_malloc(p, n);
}
int hipHostMalloc(void **p, size_t n, unsigned f)
{
    if (!pins_left) {
        ++refused;
        *p = nullptr;
        return 2;
    }
    if (pins_left > 0) --pins_left;
    ++pins;
    pinned += n;
    if (n > largest) largest = n;
    return real_host(p, n, f);
}
int hipHostFree(void *p) { ++unpinned; return real_host_free(p); }
int hipStreamCreateWithFlags(void **s, unsigned f) { ++streams; return real_stream(s, f); }
int hipStreamDestroy(void *s) { ++destroyed; return real_destroy(s); }
}
"""

CHILD = r"""
import ctypes, os, sys, tempfile
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
import mantaray_amd as mr
from mantaray_amd import _capi as C
lib = C.lib()
hip = ctypes.CDLL([l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l][0])
for name, fn in (("real_malloc", "hipMalloc"), ("real_host", "hipHostMalloc"),
                 ("real_host_free", "hipHostFree"), ("real_stream", "hipStreamCreateWithFlags"),
                 ("real_destroy", "hipStreamDestroy")):
    ctypes.c_void_p.in_dll(shim, name).value = ctypes.cast(getattr(hip, fn), ctypes.c_void_p).value
def var(name, t=ctypes.c_int):
    return t.in_dll(shim, name)
n = lambda: tuple(var(k).value for k in ("streams", "pins"))
sys.path.insert(0, sys.argv[2])
from _ncfix import create_bathymetry, create_current
tmp = tempfile.mkdtemp()
bp, cp = os.path.join(tmp, "b.nc"), os.path.join(tmp, "c.nc")
create_bathymetry(bp, 41, 31, 100.0, 100.0, lambda x, y: 50.0 + 10.0 * np.sin(x / 900.0))
create_current(cp, 41, 31, 100.0, 100.0, lambda x, y: (0.3 * np.sin(y / 800.0), 0.2 * np.cos(x / 600.0)))
one = (1500.0, 1200.0, 0.05, 0.02, 50.0, 1.0, bp, cp)
rng = np.random.default_rng(1)
def fan(rays, steps):
    ic = [rng.uniform(500.0, 2500.0, rays) for _ in range(2)] + [rng.uniform(-0.1, 0.1, rays) for _ in range(2)]
    return (*ic, float(steps), 1.0, bp, cp)
# (a process's first streams take 3 ms each: a first call makes one)
mr.core.ray_tracing(*fan(700, 900))
assert n()[0] == 1 and n()[1] > 1
C.check(lib.mr_release_host_buffers())
assert var("destroyed").value == 1 and var("unpinned").value == n()[1]
for k in ("streams", "destroyed", "pins", "unpinned"):
    var(k).value = 0
var("largest", ctypes.c_size_t).value = 0
a = mr.core.single_ray(*one)
assert n() == (1, 1) and var("largest", ctypes.c_size_t).value <= 65536, (n(), var("largest", ctypes.c_size_t).value)
calls = [fan(100, 300), fan(700, 900), fan(3000, 1000)]
first = [mr.core.ray_tracing(*c) for c in calls]
made = n()
assert var("largest", ctypes.c_size_t).value <= 4 << 20
assert 1 <= made[0] <= 12 and var("destroyed").value == 0
again = [mr.core.ray_tracing(*c) for c in calls] + [mr.core.single_ray(*one)]
assert n()[0] <= 12 and var("destroyed").value == 0
for p, q in zip(first + [a], again):
    for k in ("time", "x", "y", "kx", "ky"):
        assert np.array_equal(p[k].values, q[k].values, equal_nan=True), k
for _ in range(8):                     # up to a stream and a chunk a worker
    again = [mr.core.ray_tracing(*c) for c in calls] + [mr.core.single_ray(*one)]
made = n()
assert made[0] <= 12
for _ in range(3):
    again = [mr.core.ray_tracing(*c) for c in calls] + [mr.core.single_ray(*one)]
    for p, q in zip(first + [a], again):
        for k in ("time", "x", "y", "kx", "ky"):
            assert np.array_equal(p[k].values, q[k].values, equal_nan=True), k
assert n() == made, (n(), made)
print("kept ok", flush=True)
# all of it released
C.check(lib.mr_release_host_buffers())
assert var("destroyed").value == n()[0] and var("unpinned").value == n()[1]
print("released ok", flush=True)
# pinned memory for two workers only
var("pins_left").value = 2
got = mr.core.ray_tracing(*calls[2])
assert var("refused").value > 0
for k in ("time", "x", "y", "kx", "ky"):
    assert np.array_equal(first[2][k].values, got[k].values, equal_nan=True), k
var("pins_left").value = -1
print("few workers ok", flush=True)
# a device allocation refused once: the idle buffers go, and it is made
b, c = mr.Bathymetry.from_netcdf(bp), mr.Current.from_netcdf(cp)
before = var("unpinned").value
var("refused").value, var("refuse_once").value = 0, 1
b.upload()
assert var("refused").value == 1 and var("unpinned").value > before
print("given back ok", flush=True)
"""


def test_pool(tmp_path):
    src, so = tmp_path / "shim.cpp", str(tmp_path / "shim.so")
    src.write_text(SHIM)
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-o", so, str(src)], check=True)
    here = os.path.dirname(os.path.abspath(__file__))
    res = subprocess.run([sys.executable, "-u", "-c", CHILD, so, here], cwd=os.path.dirname(here),
                         capture_output=True, text=True, timeout=100)
    assert res.returncode == 0, res.stdout + res.stderr
    assert res.stdout.count("ok") == 4
