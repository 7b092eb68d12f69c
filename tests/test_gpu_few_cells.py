"""The PE kernels for few sub-cells (at most 8, by the tiles' half diagonal) and their
neighbours across that line, against the oracle: matrix, projections and
gradient, turned bars and elliptical holes among them."""
import numpy as np
import pytest

from conftest import TOL_FP32, assert_parity, elliptic_hole_shapes, small_geometry

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sub", [(1, 1, 1), (2, 1, 1), (1, 3, 1), (2, 1, 2), (5, 1, 1), (2, 2, 2), (3, 1, 3)])
@pytest.mark.parametrize("beta,ell", [(0.0, False), (0.3, False), (0.0, True)])
@pytest.mark.parametrize("scale", [0.5, 1.0, 2.0])  # tiles of 8 x 4 x 2 voxels: half diagonal 1.6, 3.2, 6.3 mm
def test_few_cells(smg_mod, oracle_mod, params_mod, sub, beta, ell, scale):
    p = small_geometry(params_mod, beta=beta, n_rot=3, dphi=0.4)
    p.img[3:6] = [0.8 * scale, 0.9 * scale, 1.1 * scale]
    o = oracle_mod.Oracle(p)
    shapes = elliptic_hole_shapes(9) if ell else None
    if ell:
        o.set_hole_shapes(shapes)
    ref = o.pe_matrix(rot=1, sub=sub)
    rng = np.random.default_rng(12)
    x = rng.uniform(0.5, 1.5, o.n_vox).astype(np.float32)
    y = rng.uniform(0.5, 1.5, o.n_det).astype(np.float32)
    w = rng.uniform(0.1, 1.0, ref.shape).astype(np.float32)
    with smg_mod.open_context(p) as ctx:
        if ell:
            ctx.set_hole_shapes(shapes)
        ctx.set_pe_subsamples(*sub)
        got, _ = ctx.pe_forward(1, "fp32")
        fwd, _ = ctx.pe_project(x, 1, "fp32")
        back, _ = ctx.pe_backproject(y, 1, "fp32")
        loss, grad, _ = ctx.pe_backward(w, 1, "fp32")
    what = f"{sub} beta={beta} ell={ell} scale={scale}"
    assert_parity(got, ref, TOL_FP32, "PE " + what)
    assert_parity(fwd, ref @ x.astype(np.float64), TOL_FP32, "projection " + what)
    assert_parity(back, y.astype(np.float64) @ ref, TOL_FP32, "back projection " + what)
    lref, gref = o.pe_grad(w, rot=1, sub=sub)
    assert abs(loss - lref) <= TOL_FP32 * abs(lref)
    assert np.abs(grad - gref).max() <= TOL_FP32 * np.abs(gref).max()
