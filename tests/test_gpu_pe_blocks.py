"""PE kernels at the edges of the block-wise narrowing: one sub-cell, a full
block of 64 and one past it, and candidate lists of at most 32 (several sub-cells
per pass), 33 to 64 and more than 64 (several words per sub-cell)."""
import numpy as np
import pytest

from conftest import TOL_FP32, TOL_FP64, assert_parity

pytestmark = pytest.mark.gpu


def _geometry(params_mod, layers, voxel, turn):
    p = params_mod.config(1)
    p.det[:] = 0.0
    n = layers * 9 * 9
    p.det[0] = n
    for d in range(n):
        ix, iz, il = d % 9, (d // 9) % 9, d // 81
        params_mod.set_bar(p, d, (ix - 4) * 1.5, 14.0 + 3.0 * il, (iz - 4) * 1.5, 1.5, 3.0, 1.5, res=0.10,
                           beta=turn, **params_mod.BAR_MU)
    params_mod.set_image(p, 5, 3, 3, voxel, voxel, voxel)
    return p


@pytest.mark.parametrize("layers,voxel,turn", [(1, 0.5, 0.0), (3, 2.0, 0.0), (6, 2.0, 0.0), (6, 2.0, 0.2)])
@pytest.mark.parametrize("sub", [(1, 1, 1), (4, 4, 4), (5, 13, 1), (3, 43, 1)])
def test_pe_block_edges(smg_mod, oracle_mod, params_mod, layers, voxel, turn, sub):
    p = _geometry(params_mod, layers, voxel, turn)
    o = oracle_mod.Oracle(p)
    rows = np.array([0, 13, p.n_det // 2, p.n_det - 1], np.int32)
    ref = o.pe_rows(rows, sub=sub)
    x = np.random.default_rng(3).uniform(0.0, 1.0, p.n_vox).astype(np.float32)
    with smg_mod.open_context(p) as ctx:
        ctx.set_pe_subsamples(*sub)
        for prec, tol in (("fp32", TOL_FP32), ("fp64", TOL_FP64)):
            A, st = ctx.pe_forward(0, prec)
            assert_parity(A[rows].reshape(-1), ref.reshape(-1), tol,
                          f"blocks {layers} layers {sub} {prec} fallbacks={st['fp64_fallbacks']}")
            y, _ = ctx.pe_project(x, 0, prec)
            want = A.astype(np.float64) @ x.astype(np.float64)
            # FP64 sums of the same FP32 elements, rounded once
            assert np.all(np.abs(y - want) <= 1.2e-7 * np.abs(want))


@pytest.mark.parametrize("n_bars,sub", [(81, (5, 3, 1)), (81, (4, 4, 1)), (81, (17, 1, 1)), (2048, (2, 4, 2)),
                                        (2049, (2, 4, 2))])
def test_pe_shared_items(smg_mod, oracle_mod, params_mod, n_bars, sub):
    """Items whose sub-cells several waves share (few items, 16 sub-cells and
    more), one item and one sub-cell either side of the rule, and a bar without
    attenuation.  The tangent along the matrix's mu_pe: every element is
    proportional to its bar's mu_pe, so its derivative is the element over it."""
    p = _geometry(params_mod, 1, 0.5, 0.0) if n_bars == 81 else params_mod.large_detector()
    if n_bars != 81:
        params_mod.set_image(p, 5, 3, 3, 0.5, 0.5, 0.5)
        p.det[0] = n_bars
    p.det[7 + 12 * 5] = 0.0
    o = oracle_mod.Oracle(p)
    rows = np.array([0, 5, n_bars // 2, n_bars - 1], np.int32)
    ref = o.pe_rows(rows, sub=sub)
    with smg_mod.open_context(p) as ctx:
        ctx.set_pe_subsamples(*sub)
        dmu = np.zeros(ctx._n_layers + 2 * n_bars)
        dmu[ctx._n_layers + n_bars:] = p.det[8:8 + 12 * n_bars:12]
        for prec, tol in (("fp32", TOL_FP32), ("fp64", TOL_FP64)):
            A, _ = ctx.pe_forward(0, prec)
            assert_parity(A[rows].reshape(-1), ref.reshape(-1), tol, f"shared items {n_bars} {sub} {prec}")
            dA, A2, _ = ctx.pe_tangent(dmu, 0, prec, with_matrix=True)
            assert_parity(dA[rows].reshape(-1), ref.reshape(-1), tol, f"tangent {n_bars} {sub} {prec}")
            assert_parity(A2[rows].reshape(-1), ref.reshape(-1), tol, f"tangent's matrix {n_bars} {sub} {prec}")
