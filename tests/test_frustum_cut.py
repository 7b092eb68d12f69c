"""The interval cut of the PE kernels' frustum tests, at signed zeros, denormals
and ordinary coefficients (tests/lane_frustum.cpp)."""
import ctypes as C
import itertools
import os
import subprocess

import numpy as np

from conftest import PKG, ROOT


def test_frustum_cut():
    """[lo, hi] is {s in [0, 1]: c s <= r} to the rounding of one FP32 quotient: an
    end is the exact quotient to 2^-23 of it, and the set is empty exactly where the
    rounded quotient leaves no s in [0, 1] (a quotient below the denormals is 0)."""
    out = os.path.join(ROOT, "tests", "_build")
    os.makedirs(out, exist_ok=True)
    so, src = os.path.join(out, "libfrustum.so"), os.path.join(ROOT, "tests", "lane_frustum.cpp")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wno-unknown-pragmas", "-I",
                    os.path.join(PKG, "csrc"), "-o", so, src], check=True)
    L = C.CDLL(so)
    fp = np.ctypeslib.ndpointer(np.float32, flags="C")
    L.frustum_cut_n.argtypes = [C.c_int, fp, fp, fp, fp]
    mags = [0.0, 1e-42, 1e-30, 1e-6, 0.3, 1.0, 7.0, 300.0, 1e30]
    vals = [s * m for m in mags for s in (1.0, -1.0)]
    c, r = (np.ascontiguousarray(x, np.float32) for x in zip(*itertools.product(vals, vals)))
    lo, hi = np.empty_like(c), np.empty_like(c)
    L.frustum_cut_n(len(c), c, r, lo, hi)
    def rounded(q):
        with np.errstate(over="ignore"):
            return np.float32(q)

    for ci, ri, a, b in zip(c.astype(float), r.astype(float), lo, hi):
        if ci == 0.0:
            want = (0.0, 1.0) if ri >= 0.0 else None
        elif ci > 0.0:
            want = (0.0, min(1.0, ri / ci)) if rounded(ri / ci) >= 0.0 else None
        else:
            want = (max(0.0, ri / ci), 1.0) if rounded(ri / ci) <= 1.0 else None
        if want is None:
            assert a > b, (ci, ri, a, b)
        else:
            assert a <= b, (ci, ri, a, b)
            for x, y in zip((a, b), want):
                assert abs(float(x) - y) <= 2.0 ** -23 * abs(y) + 1e-44, (ci, ri, a, b)
