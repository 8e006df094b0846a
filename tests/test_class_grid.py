"""The class grid the scoring kernels read a map through, on the CPU: the index
its tables give (tsl_check_class_grid) against the oracle's getIndex, over
points inside, on and next to every class boundary, below and above the map,
for maps of even and odd sub_dim, offsets that reach into other blocks, and
extents that end inside a block; and the maps that have no class grid."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle_binding as ob
import tsdf_localization_amd as tsl
from tsdf_localization_amd import _lib

EXACT = np.uint64(0xffffffffffffffff)

# min, extent, resolution, share of blocks allocated
MAPS = {
    "even": ((0.0, 0.0, 0.0), (6.4, 5.2, 3.2), 0.05, 0.5),
    "shifted": ((-3.7, 12.3, -1.1), (5.0, 7.3, 2.0), 0.05, 0.7),
    "chunks": ((-2.048, -4.096, 0.0), (8.192, 8.192, 4.096), 0.064, 0.6),  # 15.6 voxels a metre
    "odd": ((0.3, -0.2, 0.1), (4.0, 4.0, 4.0), 0.08, 0.8),                 # sub_dim 13
    "coarse": ((1.0, 2.0, -3.0), (9.0, 6.0, 5.0), 0.3, 0.6),
    "one": ((0.0, 0.0, 0.0), (3.0, 3.0, 3.0), 1.0, 0.5),                   # a voxel per block
    "fine": ((0.0, 0.0, 0.0), (3.0, 4.0, 3.0), 0.025, 0.6),
    "empty-top": ((0.0, 0.0, 0.0), (4.0, 4.0, 9.0), 0.1, -0.3),            # allocated near the floor only
}


def _case(name):
    lo, ext, res, share = MAPS[name]
    hi = [a + b for a, b in zip(lo, ext)]
    c = tsl.coef_init(lo, hi, res)
    rng = np.random.default_rng(sum(map(ord, name)))
    alloc = rng.uniform(size=int(c.grid_occ_size)) < abs(share)
    if share < 0:
        alloc[4 * int(c.up_dim_2):] = False
    alloc[0] = True
    sd3 = int(c.sub_dim) ** 3
    grid = np.where(alloc, (np.cumsum(alloc) - 1) * sd3, -1).astype(np.int32)
    c.data_size = int(alloc.sum()) * sd3
    return c, grid, rng


def _points(c, rng, n=15_000):
    lo = np.array([c.min_x, c.min_y, c.min_z])
    ext = np.array([c.max_x, c.max_y, c.max_z]) - lo
    res = float(c.resolution)
    p = lo + rng.uniform(-0.35, 1.35, (n, 3)) * ext
    # on and around voxel and block boundaries, the bottom band, just above it
    q = lo + np.round(rng.uniform(-1.2 / res, 1.0 / res, (n, 3)) * ext) * res
    b = lo + np.round(rng.uniform(-2, 1.2, (n, 3)) * ext)
    band = lo + rng.uniform(-1.0, 0.0, (n, 3)) * rng.integers(0, 2, (n, 3)) + rng.uniform(0, 1, (n, 3)) * ext * \
        rng.integers(0, 2, (n, 3))
    t = np.concatenate([p, q, b, band]).astype(np.float32)
    near = t.copy()
    for _ in range(2):
        t = np.concatenate([t, np.nextafter(near, np.float32(np.inf)), np.nextafter(near, np.float32(-np.inf))])
        near = np.nextafter(near, np.float32(np.inf))
    far = lo + rng.choice([-1e3, 1e3, -4e6, 4e6, 0.0], (4000, 3)) * rng.uniform(0.5, 1.0, (4000, 3))
    return np.ascontiguousarray(np.concatenate([t, far.astype(np.float32)]))


def test_maps_without_a_class_grid():
    """A voxel index that rounds up to sub_dim just below 1 m (a class a few
    floats wide), an extent past 16384 m, no allocated block."""
    has = ctypes.c_int()
    for res, ext, alloc in [(0.01, 3.0, 0), (0.02, 3.0, 0), (1.0, 17000.0, 0), (0.05, 3.0, -1)]:
        c = tsl.coef_init((0, 0, 0), (ext, 2.0, 2.0), res)
        grid = np.full(int(c.grid_occ_size), -1, np.int32)
        grid[0] = alloc
        c.data_size = int(c.sub_dim) ** 3
        _lib.check(_lib.lib.tsl_check_class_grid(ctypes.byref(c), _lib.ptr(grid), None, 0, None, ctypes.byref(has)))
        assert has.value == 0


@pytest.mark.parametrize("name", sorted(MAPS))
def test_class_grid_index_is_the_references(name):
    c, grid, rng = _case(name)
    t = _points(c, rng)
    got = np.empty(t.shape[0], np.uint64)
    has = ctypes.c_int()
    _lib.check(_lib.lib.tsl_check_class_grid(ctypes.byref(c), _lib.ptr(grid), _lib.ptr(t), t.shape[0], _lib.ptr(got),
                                             ctypes.byref(has)))
    assert has.value == 1
    # the oracle's getIndex of a point through an identity pose and scan
    om = ob.OracleMap(c, grid, np.zeros(1, np.float32))
    ref = np.array([om.get_index(*map(float, row)) for row in t], np.uint64)
    ref[ref >= c.data_size] = c.data_size
    left = got == EXACT
    assert np.array_equal(got[~left], ref[~left])
    # lanes left to the exact tiers lie below the map
    lo = np.array([c.min_x, c.min_y, c.min_z], np.float32)
    assert np.all(((t[left] - lo) <= -1.0).any(1))
    inside = ((t - lo) > -1.0).all(1)
    assert not left[inside].any()
    assert np.count_nonzero(ref[inside] < c.data_size) > 1000


@pytest.mark.parametrize("field,value", [("up_dim_2", 0), ("resolution", -1.0), ("sub_dim_2", 7), ("grid_occ_size", 0)])
def test_inconsistent_coefficients_are_refused(field, value):
    """As tsl_map_create refuses them, in a process of its own: a zero
    up_dim_2 was a division by zero."""
    code = f"""
import ctypes
import numpy as np
import tsdf_localization_amd as tsl
from tsdf_localization_amd import _lib
c = tsl.coef_init((0, 0, 0), (3, 3, 3), 0.05)
grid = np.zeros(int(c.grid_occ_size), np.int32)
c.data_size = int(c.sub_dim) ** 3
c.{field} = {value}
has = ctypes.c_int()
rc = _lib.lib.tsl_check_class_grid(ctypes.byref(c), _lib.ptr(grid), None, 0, None, ctypes.byref(has))
assert rc == _lib.TSL_ERR_INVALID_ARGUMENT, rc
"""
    r = subprocess.run([sys.executable, "-c", code], cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                       capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stderr)


def test_coordinates_out_of_range_are_left_to_the_exact_tiers():
    c, grid, _ = _case("even")
    t = np.array([[np.nan, 1, 1], [1, np.inf, 1], [1, 1, -np.inf], [4194304.0, 1, 1]], np.float32)
    got = np.zeros(4, np.uint64)
    has = ctypes.c_int()
    _lib.check(_lib.lib.tsl_check_class_grid(ctypes.byref(c), _lib.ptr(grid), _lib.ptr(t), 4, _lib.ptr(got),
                                             ctypes.byref(has)))
    assert has.value == 1 and np.all(got == EXACT)
