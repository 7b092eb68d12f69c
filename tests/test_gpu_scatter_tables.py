"""Scatter launches at the edges of the window tables: resolutions sharp enough
that the FP32 term evaluates the window probability itself, the largest and
smallest tables, windows relative to each bar's resolution, and detector
sub-cells (one batch state over several of them)."""
import numpy as np
import pytest

from conftest import TOL_FP32, TOL_FP64, assert_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res,same_window,sub", [(0.004, 1, (1, 1, 1)), (0.012, 1, (1, 1, 1)), (0.03, 0, (2, 1, 2)),
                                                 (0.1, 0, (1, 1, 1)), (0.3, 1, (1, 2, 1)), (0.9, 1, (1, 1, 1))])
def test_collimator_scatter_windows(smg_mod, oracle_mod, params_mod, res, same_window, sub):
    p = params_mod.config(3)
    params_mod.set_image(p, 9, 7, 3, 1.0, 1.0, 1.0)
    n = p.n_det
    p.det[10:10 + 12 * n:12] = np.float32(res) * np.linspace(0.97, 1.03, n).astype(np.float32)
    params_mod.set_physics(p, same_window=same_window)
    o = oracle_mod.Oracle(p)
    d, v = [a.reshape(-1).astype(np.int32) for a in np.meshgrid(np.arange(0, n, 5), np.arange(p.n_vox), indexing="ij")]
    ref = o.collimator_scatter_pairs(o.bitmap_collimator(), d, v, variant=0, sub=sub)
    assert (ref > 0).any()
    with smg_mod.open_context(p) as ctx:
        ctx.set_scatter_subsamples(*sub)
        for prec, tol in (("fp32", TOL_FP32), ("fp64", TOL_FP64)):
            got, st = ctx.scatter_collimator(0, "combined", prec)
            assert_parity(got[d, v].astype(np.float64), ref, tol,
                          f"windows res={res} same={same_window} {prec} fallbacks={st['fp64_fallbacks']}")


@pytest.mark.parametrize("n,sub", [(2, (1, 1, 1)), (32, (1, 1, 1)), (34, (1, 1, 1)), (67, (2, 1, 1)), (131, (1, 1, 1))])
def test_crystal_scatter_bitmap_words(smg_mod, oracle_mod, params_mod, n, sub):
    """Records whose bits span 1 to 6 words (several share a wave's pass), with a
    loaded bitmap that flags half of all bars, turned bars among them."""
    p = params_mod.config(4)
    params_mod.set_image(p, 5, 4, 2, 2.0, 2.0, 2.0)
    p.det[0] = n
    p.det[11:11 + 12 * n:12][1::3] = 0.3
    o = oracle_mod.Oracle(p)
    rng = np.random.default_rng(n)
    pe = rng.uniform(0, 1e-9, (n, o.n_vox)).astype(np.float32)
    bm = rng.integers(0, 1 << 32, o.bitmap_crystal().size, dtype=np.uint64).astype(np.uint32)
    d, v = [a.reshape(-1).astype(np.int32) for a in np.meshgrid(np.arange(n), np.arange(0, o.n_vox, 7), indexing="ij")]
    ref = o.crystal_scatter_pairs(pe, bm, d, v, sub=sub)
    assert (ref > 0).any()
    with smg_mod.open_context(p) as ctx:
        ctx.set_scatter_subsamples(*sub)
        ctx.load_bitmap_crystal(bm)
        for prec, tol in (("fp32", TOL_FP32), ("fp64", TOL_FP64)):
            got, _ = ctx.scatter_crystal(pe, 0, prec)
            assert_parity(got[d, v].astype(np.float64), ref, tol, f"bitmap words n={n} {prec}")


@pytest.mark.parametrize("n_rows", [1, 2, 7, 33, 64])
def test_crystal_grid_row_counts(smg_mod, params_mod, n_rows):
    """The grid points a few detector rows cannot use are left out, tested with a
    lane per (point, row): as the full matrix's rows (whose points are all
    formed), to the rounding of the different slices' sums, 2e-6 in FP32."""
    p = params_mod.config(4)
    params_mod.set_image(p, 9, 7, 1, 3.0, 3.0, 3.0)
    p.det[0] = 90
    rows = np.random.default_rng(n_rows).permutation(90)[:n_rows].astype(np.int32)
    with smg_mod.open_context(p) as ctx:
        full, _ = ctx.scatter_crystal_grid((2, 3, 2), None, 0, "fp32")
        part, _ = ctx.scatter_crystal_grid((2, 3, 2), rows, 0, "fp32")
    assert (full > 0).any()
    np.testing.assert_allclose(part, full[rows], rtol=2e-6, atol=0.0)
