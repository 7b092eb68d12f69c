"""PE elements of bars turned about y whose solid angle is the projection of an x
or z face (the reference projects those with the world direction turned by +beta,
PESysMatGen.cu:1223-1231): voxels well off the panel's axis, panels turned by
several angles, one angle per bar too."""
import math

import numpy as np
import pytest

from conftest import TOL_FP32, TOL_FP64, assert_parity, elliptic_hole_shapes
from test_lane_cpu import lane_pe

SUB = (3, 2, 3)


def panel(params_mod, turns):
    """6 x 5 bars of 2 x 8 x 2.2 mm, turned as one panel (one angle) or bar by bar
    at a wider pitch, behind a plate of 16 holes; 9 x 7 x 3 voxels of 5 mm."""
    p = params_mod.Params.empty()
    p.coll[0] = 1
    params_mod.set_layer(p, 0, 16, 90.0, 4.0, 90.0, 0.0, 0.30, 0.2, 0.1)
    for i in range(16):
        params_mod.set_hole(p, i, (i % 4 - 1.5) * 9.0, -2.0, 2.0, (i // 4 - 1.5) * 9.0, 2.0)
    p.det[0] = 30
    pitch = 2.2 if len(turns) == 1 else 3.2
    t0 = turns[0] if len(turns) == 1 else 0.0
    for k in range(30):
        x, z = (k % 6 - 2.5) * pitch, (k // 6 - 2.0) * pitch
        c, s = math.cos(t0), math.sin(t0)
        params_mod.set_bar(p, k, x * c - z * s, 14.0, x * s + z * c, 2.0, 8.0, 2.2, 0.25, 0.18, 0.07, 0.1,
                           turns[k % len(turns)])
    params_mod.set_image(p, 9, 7, 3, 5.0, 5.0, 5.0, n_rot=8, dphi=0.4, fov2coll=30.0)
    params_mod.set_physics(p)
    return p


CASES = [((0.3,), 0), ((-0.7,), 2), ((1.4,), 0), ((0.2, -0.5, 0.0, 1.1), 1)]


@pytest.mark.parametrize("turns,rot", CASES)
@pytest.mark.parametrize("exact", [0, 1])
def test_lane_turned_faces(lane_lib, oracle_mod, params_mod, turns, rot, exact):
    p = panel(params_mod, turns)
    o = oracle_mod.Oracle(p)
    d, v = (a.ravel() for a in np.meshgrid(np.arange(o.n_det), np.arange(o.n_vox), indexing="ij"))
    got, fb = lane_pe(lane_lib, p, d, v, SUB, exact, rot)
    assert_parity(got, o.pe_pairs(d, v, rot=rot, sub=SUB), TOL_FP64 if exact else TOL_FP32,
                  f"lane PE turned {turns} exact={exact} fallbacks={fb}")


@pytest.mark.gpu
@pytest.mark.parametrize("turns,rot", CASES)
@pytest.mark.parametrize("ell", [False, True])
@pytest.mark.parametrize("prec,tol", [("fp32", TOL_FP32), ("fp64", TOL_FP64)])
def test_gpu_turned_faces(smg_mod, oracle_mod, params_mod, turns, rot, ell, prec, tol):
    p = panel(params_mod, turns)
    o = oracle_mod.Oracle(p)
    shapes = elliptic_hole_shapes(o.n_holes_l0) if ell else None
    if ell:
        o.set_hole_shapes(shapes)
    ref = o.pe_matrix(rot=rot, sub=SUB)
    x = np.random.default_rng(3).uniform(0.5, 1.5, o.n_vox).astype(np.float32)
    y = np.random.default_rng(4).uniform(0.5, 1.5, o.n_det).astype(np.float32)
    with smg_mod.open_context(p) as ctx:
        if ell:
            ctx.set_hole_shapes(shapes)
        ctx.set_pe_subsamples(*SUB)
        got, _ = ctx.pe_forward(rot, prec)
        fwd, _ = ctx.pe_project(x, rot, prec)
        back, _ = ctx.pe_backproject(y, rot, prec)
    assert_parity(got, ref, tol, f"PE turned {turns} ell={ell} {prec}")
    assert_parity(fwd, ref @ x.astype(np.float64), tol, f"projection turned {turns} {prec}")
    assert_parity(back, y.astype(np.float64) @ ref, tol, f"back projection turned {turns} {prec}")
