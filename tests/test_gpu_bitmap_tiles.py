"""Bitmaps at the edges of the kernel's tiles: 64 bars per wave, 4 origins, 8
bars per store, whole and shared words, several bars at one place; and the small
ones that are built without tables (to 322 bars, to 8.4M collimator bits)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,holes", [(1, 1), (3, 2), (32, 5), (33, 4), (63, 9), (64, 3), (65, 1), (96, 6), (161, 7),
                                     (323, 100), (330, 78), (352, 70), (384, 60)])
def test_bitmaps_bit_exact(smg_mod, oracle_mod, params_mod, n, holes):
    p = params_mod.config(4)
    p.det[0], p.coll[10] = n, holes
    if n > 40:
        for c in range(1, 4):
            p.det[c + 12 * 17], p.det[c + 12 * 30] = p.det[c + 12 * 5], p.det[c + 12 * 5]
    o = oracle_mod.Oracle(p)
    with smg_mod.open_context(p) as ctx:
        for _ in range(2):  # the second over the first's words
            assert np.array_equal(ctx.bitmap_crystal(), o.bitmap_crystal())
            assert np.array_equal(ctx.bitmap_collimator(), o.bitmap_collimator())
