"""Bar-centre scatter with more pair records than one launch holds: the rows go in
chunks (128 of 512 here), in bounded memory, each row as the oracle has it."""
import numpy as np
import pytest

from conftest import TOL_FP32, TOL_FP64, assert_parity

pytestmark = pytest.mark.gpu

SUB = (4, 16, 4)
N = 512


def geometry(params_mod):
    p = params_mod.config(1)
    p.det[:] = 0.0
    p.det[0] = N
    for d in range(N):
        params_mod.set_bar(p, d, (d % 16 - 7.5) * 2.1, 17.5 + 10.5 * (d // 256), (d // 16 % 16 - 7.5) * 2.1, 2.0, 10.0,
                           2.0, res=0.1, **params_mod.BAR_MU)
    params_mod.set_image(p, 3, 2, 2, 8.0, 8.0, 8.0)
    params_mod.set_physics(p, lo=90.0, hi=154.55)
    return p


def test_rows_in_chunks(smg_mod, oracle_mod, params_mod):
    import torch
    p = geometry(params_mod)
    o = oracle_mod.Oracle(p)
    pe = np.random.default_rng(8).uniform(0, 1e-9, (N, o.n_vox)).astype(np.float32)
    bm = o.bitmap_crystal()
    got = {}
    with smg_mod.open_context(p) as ctx:
        ctx.build_bitmap()
        free0 = torch.cuda.mem_get_info(0)[0]
        ctx.set_scatter_subsamples(*SUB)
        for prec in ("fp32", "fp64"):
            got[prec] = ctx.scatter_crystal(pe, 0, prec)[0]
        grown = free0 - torch.cuda.mem_get_info(0)[0]
    records = N * N * SUB[0] * SUB[1] * SUB[2]
    print(f"{records} records, {grown / 2**20:.0f} MiB", flush=True)
    assert grown <= 48 * records  # the sums of the chords alone for all of them
    assert (got["fp64"] > 0).mean() > 0.5
    assert_parity(got["fp32"], got["fp64"], TOL_FP32, "rows in chunks, FP32 against FP64")
    d = np.array([0, 127, 128, 255, 256, 511], np.int32)  # the chunks' ends
    v = np.array([0, 5, 11, 3, 7, 10], np.int32)
    ref = o.crystal_scatter_pairs(pe, bm, d, v, sub=SUB)
    for prec, tol in (("fp32", TOL_FP32), ("fp64", TOL_FP64)):
        assert_parity(got[prec][d, v], ref, tol, f"rows in chunks {prec}")
