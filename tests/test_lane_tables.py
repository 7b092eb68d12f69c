"""The scatter kernels' tables, built for the host (tests/lane_tables.cpp): KN
prefix polynomials, window probabilities, and the FP32 angle."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from conftest import PKG, ROOT


@pytest.fixture(scope="module")
def tables_lib():
    out = os.path.join(ROOT, "tests", "_build")
    os.makedirs(out, exist_ok=True)
    so, src = os.path.join(out, "libtables.so"), os.path.join(ROOT, "tests", "lane_tables.cpp")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wno-unknown-pragmas", "-I",
                    os.path.join(PKG, "csrc"), "-o", so, src], check=True)
    L = C.CDLL(so)
    fp = np.ctypeslib.ndpointer(np.float32, flags="C")
    ip = np.ctypeslib.ndpointer(np.int32, flags="C")
    dp = np.ctypeslib.ndpointer(np.float64, flags="C")
    L.table_kn_sums.argtypes = [C.c_double, dp, dp, C.c_int, dp]
    L.table_window.argtypes = [C.c_double] * 4 + [dp, C.c_int, dp, dp, ip, ip]
    L.table_angles.argtypes = [fp, fp, C.c_int, fp]
    return L


@pytest.mark.parametrize("e0", [30.0, 140.5, 511.0])
def test_kn_polynomial_sums(tables_lib, oracle_mod, e0):
    """The polynomials' sums equal the oracle's node-by-node sums (scatter.cu:
    980-993): prefix sums up to ~2 held to a few FP64 roundings, so 5e-15
    absolute, and 1e-11 relative on the smallest sums (one node near 0 rad)."""
    rng = np.random.default_rng(5)
    lo = rng.uniform(0.0, 3.1, 3000)
    hi = np.minimum(lo + rng.exponential(0.1, 3000), np.pi)
    lo[:100], hi[100:200] = 0.0, np.pi
    lo[200:260] = np.arange(60) * float(np.float32(0.01))  # on and next to a node
    lo[260:300] = np.nextafter(lo[200:240], 4.0)
    hi[200:300] = lo[200:300] + 0.0234
    out = np.zeros(len(lo))
    tables_lib.table_kn_sums(e0, lo, hi, len(lo), out)
    ref = np.array([oracle_mod.kn_sum(e0, a, b, float(np.float32(0.01))) for a, b in zip(lo, hi)])
    err = np.abs(out - ref)
    print(f"KN polynomials e0={e0}: max abs {err.max():.1e}, max rel {(err / np.maximum(ref, 1e-5)).max():.1e}")
    assert err.max() <= 5e-15 and np.all(err <= 1e-11 * np.maximum(ref, 1e-5))


@pytest.mark.parametrize("e0,lo,hi", [(140.5, 126.45, 154.55), (140.5, 100.0, 135.0), (140.5, 60.0, 300.0),
                                      (364.0, 328.0, 400.0), (511.0, 435.0, 650.0)])
@pytest.mark.parametrize("res", [0.015, 0.03, 0.1, 0.3])
def test_window_table(tables_lib, e0, lo, hi, res):
    """The row table against the direct probability: the cubics' 2e-8 and a few
    FP32 roundings (coefficients and evaluation, below 3e-7 together), and the
    2-sigma cuts by limits on 1 - cos(theta) as the reference's tests make them."""
    rng = np.random.default_rng(6)
    omc = np.concatenate([rng.uniform(0.0, 2.0, 20000), rng.exponential(0.05, 2000) % 2.0, [0.0, 2.0, 1e-12]])
    tab, direct = np.zeros(len(omc)), np.zeros(len(omc))
    p1, p2 = np.zeros(len(omc), np.int32), np.zeros(len(omc), np.int32)
    n = tables_lib.table_window(e0, lo, hi, res, omc, len(omc), tab, direct, p1, p2)
    if n == 0:
        assert res < 0.05  # the direct form takes over
        return
    assert np.array_equal(p1, p2)
    ok = p1 != 0
    if ok.any():
        rel = np.abs(tab[ok] - direct[ok]) / direct[ok]
        print(f"window table e0={e0} [{lo}, {hi}] res={res}: {n} intervals, max rel {rel.max():.1e}")
        assert rel.max() <= 3.2e-7


def test_angle_fp32(tables_lib):
    """angle_f against atan2 in FP64 over [0, pi], small angles included: the fit's
    1.5e-8 and about six FP32 roundings."""
    rng = np.random.default_rng(7)
    th = np.concatenate([rng.uniform(0, np.pi, 20000), 10.0 ** rng.uniform(-6, 0, 20000), [0.0, np.pi / 2, np.pi]])
    s, c = np.sin(th).clip(0).astype(np.float32), np.cos(th).astype(np.float32)
    out = np.zeros(len(th), np.float32)
    tables_lib.table_angles(s, c, len(th), out)
    ref = np.arctan2(s.astype(np.float64), c.astype(np.float64))
    err = np.abs(out - ref) / np.maximum(ref, 1e-30)
    assert err.max() <= 4e-7
