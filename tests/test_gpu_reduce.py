"""The scan reduction's hash table and counting passes, bit for bit the
oracle's: one point to more than the 256 x 1024 of one tile per workgroup,
points all in one cell, all in cells of their own, and a few to a cell."""
import numpy as np
import pytest

import oracle_binding as ob

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spread", [0.0, 0.3, 30.0])
@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 2049, 262144, 300001])
def test_reduction_sizes(n, spread):
    import tsdf_localization_amd as tsl
    from tsdf_localization_amd import synth
    room = synth.room()
    f = tsl.DeviceFilter(tsl.TSDFEvaluator(room.map), 16)
    rng = np.random.default_rng(n)
    pts = (rng.normal(0, 1, (n, 3)) * spread + 2.0).astype(np.float32)
    pts[::5] *= np.float32(0.1)  # some closer than 1 m
    rings = rng.integers(0, 64, n)
    f.set_scan_raw(pts, rings.astype(np.int16), room.tf, 0.064)
    got, ref = f.get_scan(), ob.reduce_scan(pts, rings, 0.064)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
    for shift in (0, -40, 70000):  # low bytes only, and rings of more than 8 bits
        r = (rings + shift * (rings > 30)).astype(np.int32)
        f.set_scan_cloud(pts, r, room.tf)
        got, ref = f.get_scan(), ob.reduce_cloud(pts, r)
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), shift
