"""What the cell records hold of an axis (mantaray_amd/csrc/mr_axes.h, plain
C++), through a small driver built here with g++ (tests/axes/axes_driver.cpp):
the cell thresholds are bit for bit those of a bisection over every
floating-point value, every fast region lies in its cell and on no node, and
the share of a cell outside its region tells the axes that run on cell records
from those that do not.  Host code only; no GPU is involved.
"""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LINE = 1.0 / 1024                                        # half of kOutside: one of two axes


def _axes():
    """(name, f64 coordinates, whether the share is below the line in f32 and
    in f64; None where an axis is there for its thresholds alone)"""
    rng = np.random.default_rng(2)
    a = [("from zero", 100.0 * np.arange(401), True, True),
         ("thirds", 37.0 / 3.0 * np.arange(1500), True, True),
         # the first spacing's f32 rounding is 3e-4 of it, over 40 cells
         ("across zero", -1000.0 + 0.1 * np.arange(41), False, False),
         # 130 f32 values a cell, one of them on the node
         ("far, coarse in f32", 4.0e6 + 33.333 * np.arange(907), False, False),
         # the f32 rounding of the first spacing adds up over the axis
         ("first spacing off", 500000.0 + 33.333 * np.arange(1201), False, False),
         ("far, 1 km", 500000.0 + 1000.0 * np.arange(300), True, True),
         ("jittered", 40.0 * np.arange(34) + rng.uniform(-8.0, 8.0, 34), False, False),
         ("stretched", 10.0 * np.cumsum(1.01 ** np.arange(200)), False, False),
         ("descending", 2.0 - 0.7 * np.arange(12), False, False),
         ("repeated node", np.array([0.0, 10.0, 20.0, 20.0, 30.0]), False, False),
         ("two nodes", np.array([-7.0, 0.0]), True, True),
         ("far", 1.0e7 + 3.3 * np.arange(17), False, False),
         ("tiny", 3.0e-30 + 7.0e-31 * np.arange(9), None, None),
         ("subnormal", 1.0e-41 * np.arange(9), None, None),
         ("huge", -2.0e30 + 1.7e29 * np.arange(30), None, None),
         ("spacing overflows", np.array([-3.0e38, 3.0e38]), False, None),
         ("one spacing overflows", np.array([-3.4e38, -3.0e38, 3.0e38]), None, None)]
    a += [(f"random {i}", rng.normal() * 10.0 ** rng.uniform(-3, 7)
           + 10.0 ** rng.uniform(-3, 5) * np.cumsum(rng.uniform(0.5, 1.5, rng.integers(2, 60))),
           None, None) for i in range(300)]
    return a


@pytest.fixture(scope="module")
def checked(tmp_path_factory):
    """{(name, 32 or 64): (wrong thresholds, wrong regions, share)}"""
    tmp = tmp_path_factory.mktemp("axes")
    exe, data = str(tmp / "driver"), str(tmp / "axes.bin")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off",
                    "-I", os.path.join(ROOT, "mantaray_amd", "csrc"), "-o", exe,
                    os.path.join(ROOT, "tests", "axes", "axes_driver.cpp")], check=True)
    keys = []
    with open(data, "wb") as f:
        for name, a, *_ in _axes():
            for kind in (32, 64):
                v = a.astype(np.float32).astype(np.float64) if kind == 32 else a
                if v[0] == v[1]:
                    continue                             # refused: no spacing
                f.write(np.array([kind, v.size], dtype=np.int64).tobytes() + v.tobytes())
                keys.append((name, kind))
    out = subprocess.run([exe, data], check=True, capture_output=True, text=True).stdout
    rows = [ln.split() for ln in out.splitlines()]
    assert len(rows) == len(keys) > 600
    return {k: (int(r[0]), int(r[1]), float(r[2])) for k, r in zip(keys, rows)}


def test_thresholds(checked):
    assert not {k: v[0] for k, v in checked.items() if v[0]}


def test_fast_regions(checked):
    assert not {k: v[1] for k, v in checked.items() if v[1]}


def test_share_outside(checked):
    for name, _, in32, in64 in _axes():
        for kind, below in ((32, in32), (64, in64)):
            if below is not None:
                assert (checked[name, kind][2] <= LINE) == below, (name, kind, checked[name, kind])
