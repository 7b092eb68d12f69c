"""Wave-level selection of the PE kernels' candidates, built for the host
(tests/lane_tiles.cpp)."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from conftest import PKG, ROOT, elliptic_hole_shapes, narrow_plate_geometry, small_geometry


@pytest.fixture(scope="module")
def tiles_lib():
    out = os.path.join(ROOT, "tests", "_build")
    os.makedirs(out, exist_ok=True)
    so, src = os.path.join(out, "libtiles.so"), os.path.join(ROOT, "tests", "lane_tiles.cpp")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wno-unknown-pragmas", "-I",
                    os.path.join(PKG, "csrc"), "-o", so, src], check=True)
    L = C.CDLL(so)
    fp = np.ctypeslib.ndpointer(np.float32, flags="C")
    dp = np.ctypeslib.ndpointer(np.float64, flags="C")
    L.tile_extent_check.restype = C.c_int
    L.tile_extent_check.argtypes = [fp, fp, fp, fp, fp] + [C.c_int] * 9 + [C.c_uint, dp]
    L.cull_all_check.restype = C.c_int
    L.cull_all_check.argtypes = [fp, fp, fp, fp] + [C.c_int] * 5 + [C.c_uint, dp]
    return L


@pytest.mark.parametrize("case,rot,tile", [("small", 0, (8, 8, 1)), ("volume", 3, (4, 4, 4)), ("full", 0, (4, 4, 4)),
                                           ("turned", 1, (8, 4, 2)), ("close", 0, (8, 8, 1))])
def test_cull_keeps_all_is_conservative(tiles_lib, params_mod, case, rot, tile):
    """A candidate kept for a whole tile at once passes the reference culling test
    of each of its voxels; "close": voxels of 6 mm next to the plate, where the
    tile is large against its distance."""
    if case == "full":
        p = params_mod.config(2)
    elif case == "turned":
        p = small_geometry(params_mod, beta=0.4, nx=9, ny=9, nz=2, dphi=0.3, n_rot=3)
    else:
        p = params_mod.config(1)
        dims, w = {"small": ((19, 13, 1), 1.0), "volume": ((10, 9, 7), 1.1), "close": ((9, 9, 1), 6.0)}[case]
        params_mod.set_image(p, *dims, w, w, w, 12, 0.31)
    st = np.zeros(3)
    assert tiles_lib.cull_all_check(p.coll, p.det, p.img, p.phys, rot, *tile, 20, 11, st) == 0
    print(f"{case}: {int(st[0])} of {int(st[2])} fully kept candidates found at once")
    assert st[0] > 0 and st[1] == 0


@pytest.mark.parametrize("case,rot,tile,sub,waves", [
    ("flat", 0, (8, 8, 1), (2, 3, 2), 12),       # one slice: no extent along z
    ("flat", 5, (8, 8, 1), (2, 3, 2), 12),       # turned about z by an odd angle
    ("thin", 2, (8, 4, 2), (2, 3, 2), 12),
    ("volume", 0, (4, 4, 4), (3, 1, 2), 12),
    ("volume", 3, (4, 4, 4), (3, 1, 2), 12),
    ("turned", 1, (8, 4, 2), (2, 2, 2), 12),     # bars turned about y
    ("plates", 2, (8, 4, 2), (2, 2, 2), 12),     # three plates, turned bars
    ("narrow", 1, (8, 4, 2), (2, 2, 2), 12),
    ("ellipses", 4, (8, 8, 1), (2, 3, 2), 12),
    ("voxel", 0, (8, 8, 1), (2, 4, 2), 60),       # a single voxel: no extent at all
])
def test_tile_extents_drop_no_chord(tiles_lib, params_mod, case, rot, tile, sub, waves):
    """No bar or hole with a chord above 0 on any ray of a tile is dropped by the
    tile test or the sub-cell test with the tile's box extents, and the extents
    keep no more pairs than the bounding ball (up to its rounding margin)."""
    shapes = np.zeros(0, np.float32)
    if case in ("flat", "ellipses", "voxel"):
        p = params_mod.config(1)
        params_mod.set_image(p, *((1, 1, 1) if case == "voxel" else (19, 13, 1)), 1.0, 0.8, 1.0, 12, 0.31)
        if case == "ellipses":
            shapes = np.ascontiguousarray(elliptic_hole_shapes(p.n_holes), np.float32).reshape(-1)
    elif case == "thin":
        p = params_mod.config(1)
        params_mod.set_image(p, 13, 9, 2, 1.1, 0.9, 1.3, 12, 0.31)
    elif case == "volume":
        p = params_mod.config(1)
        params_mod.set_image(p, 10, 9, 7, 1.1, 0.9, 1.3, 12, 0.31)
    elif case == "turned":
        p = small_geometry(params_mod, beta=0.4, nx=9, ny=9, nz=2, dphi=0.3, n_rot=3)
    elif case == "plates":
        p = small_geometry(params_mod, beta=0.05, layers=3, dphi=0.3, n_rot=3)
    else:
        p = narrow_plate_geometry(params_mod)
    st = np.zeros(6)
    assert tiles_lib.tile_extent_check(p.coll, p.det, p.img, p.phys, shapes, len(shapes) // 3, rot, *sub, *tile,
                                       waves, 7, st) == 0
    print(f"{case}: {int(st[0])} chords; pairs kept {int(st[3])}, with the ball {int(st[4])}")
    assert st[0] > 0
    assert st[1] == 0 and st[2] == 0
    assert st[3] <= st[4] and st[5] == 0
