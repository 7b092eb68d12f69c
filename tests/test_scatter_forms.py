"""The scatter term in each form the kernels have: FP64, FP32 with the row's window
table, and FP32 with the window probability per term (wide windows and sharp
resolutions, which have no table).  All three take their KN sums from the prefix
polynomials."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from conftest import PKG, ROOT, TOL_FP32, TOL_FP64, assert_parity

NARROW = dict(lo=126.45, hi=154.55, e0=140.5)
SHARP = dict(lo=90.0, hi=154.55, e0=140.5)
WIDE = dict(lo=250.0, hi=650.0, e0=511.0)


def geometry(params_mod, window, res):
    p = params_mod.config(3)
    params_mod.set_physics(p, **window)
    for d in range(p.n_det):
        p.det[12 * d + 10] = res
    return p


@pytest.fixture(scope="module")
def forms_lib():
    out = os.path.join(ROOT, "tests", "_build")
    os.makedirs(out, exist_ok=True)
    so = os.path.join(out, "libforms.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wno-unknown-pragmas", "-I",
                    os.path.join(PKG, "csrc"), "-o", so, os.path.join(ROOT, "tests", "lane_forms.cpp")], check=True)
    L = C.CDLL(so)
    fp = np.ctypeslib.ndpointer(np.float32, flags="C")
    ip = np.ctypeslib.ndpointer(np.int32, flags="C")
    dp = np.ctypeslib.ndpointer(np.float64, flags="C")
    up = np.ctypeslib.ndpointer(np.uint32, flags="C")
    L.form_scatter_pairs.restype = C.c_long
    L.form_scatter_pairs.argtypes = [fp] * 5 + [up] + [C.c_int] * 7 + [ip, ip, C.c_int, dp]
    L.form_row_intervals.argtypes = [C.c_double] * 4
    L.form_launch_intervals.argtypes = [C.c_double] * 3 + [C.c_int] + [C.c_double] * 2
    return L


@pytest.mark.parametrize("kind,variant,sub", [(0, 0, (1, 1, 1)), (1, 0, (1, 1, 1)), (1, 1, (2, 1, 2))])
@pytest.mark.parametrize("window,res", [(NARROW, 0.1), (SHARP, 0.005), (WIDE, 0.1)])
@pytest.mark.parametrize("form", [0, 1, 2])
def test_lane_forms(forms_lib, oracle_mod, params_mod, kind, variant, sub, window, res, form):
    p = geometry(params_mod, window, res)
    o = oracle_mod.Oracle(p)
    rng = np.random.default_rng(31 + kind)
    pe = rng.uniform(0, 1e-9, (o.n_det, o.n_vox)).astype(np.float32)
    bm = o.bitmap_crystal() if kind == 0 else o.bitmap_collimator()
    d = rng.integers(0, o.n_det, 150).astype(np.int32)
    v = rng.integers(0, o.n_vox, 150).astype(np.int32)
    out = np.zeros(150)
    fb = forms_lib.form_scatter_pairs(p.coll, p.det, p.img, p.phys, pe, bm, kind, variant, 0, *sub, form, d, v, 150,
                                      out)
    if form == 1 and out[0] == -1.0:
        assert window is WIDE or res < 0.02  # no table: the third form serves
        return
    ref = (o.crystal_scatter_pairs(pe, bm, d, v, sub=sub) if kind == 0
           else o.collimator_scatter_pairs(bm, d, v, variant=variant, sub=sub))
    assert (ref > 0).any() and fb >= 0
    assert_parity(out, ref, TOL_FP32 if form else TOL_FP64, f"form {form} kind={kind} res={res} fallbacks={fb}")


@pytest.mark.parametrize("e0,lo,hi,same", [(140.5, 0, 0, 0), (511.0, 0, 0, 0), (140.5, 126.45, 154.55, 1),
                                           (364.0, 200.0, 300.0, 1), (511.0, 350.0, 650.0, 1)])
@pytest.mark.parametrize("res_lo,res_hi", [(0.1, 0.77), (0.09, 0.11), (0.05, 0.05), (0.012, 0.5)])
def test_launch_intervals(forms_lib, e0, lo, hi, same, res_lo, res_hi):
    """A launch's window tables have the intervals that each of its rows needs
    (kWinStep), and no tables where a row has none; the need between the steps of
    1.25 in the resolution is within one doubling only next to a step."""
    n = forms_lib.form_launch_intervals(e0, lo, hi, same, res_lo, res_hi)
    ends = []
    for r in np.geomspace(res_lo, res_hi, 40):
        a, b = (lo, hi) if same else ((1 - r / 2) * e0, (1 + r / 2) * e0)
        ends.append(forms_lib.form_row_intervals(e0, a, b, r))
    assert (n == 0) == (min(ends) == 0)
    if n:
        assert n == max(ends)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["crystal", "collimator", "grid", "crystal_grid"])
def test_gpu_bar_without_attenuation(smg_mod, params_mod, kind):
    """A bar without attenuation has no terms, so its resolution does not change how
    the other rows are formed."""
    out = []
    for res in (0.1, 0.0):
        p = params_mod.config(1)
        params_mod.set_image(p, 16, 16, 2, 2.0, 2.0, 2.0)
        p.det[12 * 5 + 7:12 * 5 + 11] = [0.0, 0.0, 0.0, res]
        pe = np.random.default_rng(5).uniform(0, 1e-9, (p.n_det, p.n_vox)).astype(np.float32)
        with smg_mod.open_context(p) as ctx:
            if kind == "crystal":
                got = ctx.scatter_crystal(pe, 0, "fp32")[0]
            elif kind == "collimator":
                got = ctx.scatter_collimator(0, "combined", "fp32")[0]
            elif kind == "grid":
                got = ctx.scatter_collimator_grid(4.0, 0, "fp32")[0]
            else:
                got = ctx.scatter_crystal_grid((2, 2, 2), np.array([3, 5, 9]), 0, "fp32")[0]
        out.append(got)
    assert (out[0] > 0).any()
    assert np.array_equal(out[0], out[1])


@pytest.mark.gpu
@pytest.mark.parametrize("window,res", [(NARROW, 0.1), (SHARP, 0.005), (WIDE, 0.1)])
@pytest.mark.parametrize("kind", ["crystal", "collimator", "grid"])
def test_gpu_forms(smg_mod, params_mod, window, res, kind):
    """FP32 against FP64 for windows with a table and without; the KN node count
    sends no term to FP64 in either form (formed in FP32 alone it is in doubt for 4
    in 10,000 of the terms inside the window)."""
    p = geometry(params_mod, window, res)
    pe = np.random.default_rng(5).uniform(0, 1e-9, (p.n_det, p.n_vox)).astype(np.float32)
    out = {}
    with smg_mod.open_context(p) as ctx:
        for prec in ("fp32", "fp64"):
            if kind == "crystal":
                out[prec] = ctx.scatter_crystal(pe, 0, prec)[:2]
            elif kind == "collimator":
                out[prec] = ctx.scatter_collimator(0, "combined", prec)[:2]
            else:
                out[prec] = ctx.scatter_collimator_grid(4.0, 0, prec)[:2]
    got, ref = out["fp32"][0], out["fp64"][0]
    st = out["fp32"][1]
    assert (ref > 0).any()
    assert_parity(got, ref, TOL_FP32, f"{kind} {window} res={res} fallbacks={st['fp64_fallbacks']} of {st['rays']}")
    assert st["fp64_fallbacks"] <= 1e-5 * st["rays"]
