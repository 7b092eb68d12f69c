"""The bitmap kernel's FP32 decisions (tests/lane_bitmap.cpp) against the
reference's test in FP64."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from conftest import PKG, ROOT


@pytest.fixture(scope="module")
def bitmap_lib():
    out = os.path.join(ROOT, "tests", "_build")
    os.makedirs(out, exist_ok=True)
    so, src = os.path.join(out, "libbitmap.so"), os.path.join(ROOT, "tests", "lane_bitmap.cpp")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wno-unknown-pragmas", "-I",
                    os.path.join(PKG, "csrc"), "-o", so, src], check=True)
    L = C.CDLL(so)
    L.bitmap_decisions.argtypes = [np.ctypeslib.ndpointer(np.float64, flags="C"), C.c_int, C.c_int,
                                   C.POINTER(C.c_long), C.POINTER(C.c_long), C.POINTER(C.c_double)]
    return L


@pytest.mark.parametrize("coll", [0, 1])
@pytest.mark.parametrize("kind", ["far", "touching", "grid", "coincident", "points"])
def test_bitmap_decisions(bitmap_lib, coll, kind):
    """Every decision outside the band equals FP64's; a margin near 0 is off by
    at most 36 units of 2^-24 (the sum of its roundings), three quarters of the
    band.  Random centres 100 mm away with radii from a tenth to a hundredth of
    their distances, spheres that touch, the ties of a regular grid, several
    bars at one place, and radii of 0."""
    rng = np.random.default_rng(3)
    s = np.zeros((150, 4))
    s[:, :3] = np.float32(rng.uniform(-60, 60, (150, 3)) + [0, 120, 0])
    s[:, 3] = rng.uniform(0.3, 6, 150)
    if kind == "touching":
        s[:, :3] = np.float32(rng.uniform(-6, 6, (150, 3)))
    elif kind == "grid":
        g = np.stack(np.meshgrid(np.arange(10), np.arange(3), np.arange(5), indexing="ij"), -1).reshape(-1, 3)
        s[:, :3], s[:, 3] = 2.0 * g + [0, 17.5, 0], 1.0
    elif kind == "coincident":
        s[40:60, :3] = s[20:40, :3]
        s[60:70, :3] = s[20:30, :3]
    elif kind == "points":
        s[:, 3] = 0.0
    wrong, left, err = C.c_long(), C.c_long(), C.c_double()
    bitmap_lib.bitmap_decisions(np.ascontiguousarray(s), 150, coll, wrong, left, err)
    print(f"{kind}: left to FP64 {left.value}, largest error {err.value * 2**24:.1f} * 2^-24")
    assert wrong.value == 0
    assert err.value <= 36 * 2.0 ** -24
