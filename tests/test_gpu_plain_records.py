"""Traces on the plain records, where a field has no cell records of its own:
the form of the kernel is that of the rows wanted (all four arrays, none, or
any subset; the last one tests each array in every step), and every form gives
the rows of a trace on cell records bitwise.

The fields come to their plain records in a child process in which hipMalloc
refuses anything as large as the own records; the kernels launched are read
off hipLaunchKernel there.  Both are definitions that stand before the
runtime's.
"""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

SHIM = r"""
#include <cstddef>
#include <cstring>
#include <dlfcn.h>
struct dim3 {
    unsigned x, y, z;
};
extern "C" {
int (*real_malloc)(void **, size_t) = nullptr;
int (*real_launch)(const void *, dim3, dim3, void **, size_t, void *) = nullptr;
size_t limit = 0;                      // 0: none
char last[512];                        // the last kernel launched
int hipMalloc(void **p, size_t n)
{
    if (limit && n >= limit) {
        *p = nullptr;
        return 2;                      // hipErrorOutOfMemory
    }
    return real_malloc(p, n);
}
int hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t lds, void *stream)
{
    Dl_info i;
    last[0] = 0;
    if (dladdr(f, &i) && i.dli_sname) std::strncpy(last, i.dli_sname, sizeof last - 1);
    return real_launch(f, g, b, args, lds, stream);
}
}
"""

CHILD = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
import mantaray_amd as mr
from mantaray_amd import _capi as C
lib = C.lib()
hip = ctypes.CDLL([l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l][0])
for name, fn in (("real_malloc", hip.hipMalloc), ("real_launch", hip.hipLaunchKernel)):
    ctypes.c_void_p.in_dll(shim, name).value = ctypes.cast(fn, ctypes.c_void_p).value
limit = ctypes.c_size_t.in_dll(shim, "limit")
last = (ctypes.c_char * 512).in_dll(shim, "last")
sys.path.insert(0, sys.argv[2])
from test_gpu_upload import PAIRS, _fields, _rays
N, NR, DT = 700, 130, 0.7
rays = [np.ascontiguousarray(v) for v in _rays(NR)]
rays[0][:3] = 40.0 * N * 1.2                             # off the grid: ended rays
def trace(b, c, steps, keep, math):
    r = {k: np.full((steps + 1, NR), 7.0) for k in ("x", "y", "kx", "ky")}
    r["len"], r["end"] = np.zeros(NR, np.int32), np.zeros((NR, 4))
    o = C.options(math=math)
    C.check(lib.mr_trace_many(b.handle, c.handle, NR, *[v.ctypes.data for v in rays], 0.0,
                              steps * DT, DT, ctypes.byref(o), None,
                              *[r[k].ctypes.data if k in keep else None
                                for k in ("x", "y", "kx", "ky")],
                              r["len"].ctypes.data, r["end"].ctypes.data))
    return r
for pair in PAIRS:
    b, c = _fields(pair, N)
    limit.value = 699 * 699 * (64 if pair == "depth only" else 128) - 1000
    pb, pc = _fields(pair, N)
    for math in (C.MR_MATH_FAST, C.MR_MATH_LITERAL):
        for steps, keep in ((1, "x y kx ky"), (37, "x y kx ky"), (37, ""), (37, "y kx")):
            keep = keep.split()
            limit.value, lim = 0, limit.value
            want = trace(b, c, steps, keep, math)
            limit.value = lim
            got = trace(pb, pc, steps, keep, math)
            for k, v in want.items():
                assert np.array_equal(got[k], v, equal_nan=True), (pair, steps, keep, k)
            bk, ck = ("1" if pair == "current only" else "3"), ("0" if pair == "depth only" else "1")
            out = {4: 1, 0: 0}.get(len(keep), 2)
            want = f"trace_kernelILi{bk}ELi{ck}ELi{math}ELi{out}ELi0ELb0EE"
            assert want in last.value.decode(), (want, last.value)
    limit.value = 0
    print(pair, "ok", flush=True)
"""


def test_forms_of_the_plain_route(tmp_path):
    src, so = tmp_path / "shim.cpp", str(tmp_path / "shim.so")
    src.write_text(SHIM)
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-o", so, str(src), "-ldl"], check=True)
    here = os.path.dirname(os.path.abspath(__file__))
    res = subprocess.run([sys.executable, "-u", "-c", CHILD, so, here], cwd=os.path.dirname(here),
                         capture_output=True, text=True, timeout=100)
    assert res.returncode == 0, res.stdout + res.stderr
    assert res.stdout.count("ok") == 3
