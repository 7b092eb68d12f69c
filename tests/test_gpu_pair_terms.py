"""The pair terms with few and many records a wave (8 to 64, by their number): crystal
and collimator scatter of detectors of 5 to 400 bars, 1 to 12 sub-cells, against the
oracle."""
import numpy as np
import pytest

from conftest import TOL_FP32, TOL_FP64, assert_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bars,sub", [(5, (1, 1, 1)), (33, (1, 3, 1)), (130, (1, 1, 1)), (130, (2, 3, 2)),
                                      (400, (1, 1, 1))])
@pytest.mark.parametrize("turn", [0.0, 0.2])
def test_records_per_wave(smg_mod, oracle_mod, params_mod, bars, sub, turn):
    p = params_mod.config(1)
    p.det[:] = 0.0
    p.det[0] = bars
    for d in range(bars):
        params_mod.set_bar(p, d, (d % 10 - 4.5) * 2.6, 17.5 + 13.0 * (d // 100), (d // 10 % 10 - 4.5) * 2.6, 2.0, 10.0,
                           2.0, res=0.1, beta=turn, **params_mod.BAR_MU)
    params_mod.set_image(p, 5, 4, 1, 6.0, 6.0, 6.0)
    params_mod.set_physics(p, lo=80.0, hi=154.55)
    o = oracle_mod.Oracle(p)
    pe = np.random.default_rng(8).uniform(0, 1e-9, (bars, o.n_vox)).astype(np.float32)
    bc, bh = o.bitmap_crystal(), o.bitmap_collimator()
    rng = np.random.default_rng(9)
    d = rng.integers(0, bars, 60).astype(np.int32)
    v = rng.integers(0, o.n_vox, 60).astype(np.int32)
    with smg_mod.open_context(p) as ctx:
        ctx.set_scatter_subsamples(*sub)
        for prec, tol in (("fp32", TOL_FP32), ("fp64", TOL_FP64)):
            got = ctx.scatter_crystal(pe, 0, prec)[0]
            ref = o.crystal_scatter_pairs(pe, bc, d, v, sub=sub)
            assert (ref > 0).any()
            assert_parity(got[d, v], ref, tol, f"crystal {bars} bars {sub} {prec}")
            got = ctx.scatter_collimator(0, "combined", prec)[0]
            ref = o.collimator_scatter_pairs(bh, d, v, variant=0, sub=sub)
            assert (ref > 0).any()
            assert_parity(got[d, v], ref, tol, f"collimator {bars} bars {sub} {prec}")
