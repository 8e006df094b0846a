"""Maps without a class grid, scored by the kernels that form the reference's
index per pair: bricked and linear voxels, block offsets from the rank table
and from the block table, block strides past 24 bits, palette and float form.
Values bit for bit the oracle's, weights within 1e-5 of its float64 sum (at
most N / 64 + 6 + chunks float additions of non-negative terms, 2^-24 each), the
same bits for every tile shape, particle order and block lookup, and for a
batch's member as alone."""
import ctypes

import numpy as np
import pytest

import oracle_binding as ob
from test_gpu_parity import WEIGHT_RTOL, oracle_values, rel_err

pytestmark = pytest.mark.gpu

# extent, resolution
MAPS = {
    "bricked": ((3.0, 3.0, 1.0), 0.01),     # sub_dim 100
    "linear": ((4.0, 4.0, 3.0), 0.04),      # sub_dim 25
    "even": ((4.0, 3.0, 2.0), 0.02),        # sub_dim 50, linear
    "long": ((420.0, 3.0, 2.0), 0.05),      # bucket tables past the LDS
    "strides": ((4096.0, 2100.0, 1.0), 0.25),  # up_dim_2 past 2^23
}
CHUNK = 128


def _setup(name, form):
    import tsdf_localization_amd as tsl
    from tsdf_localization_amd import _lib
    ext, res = MAPS[name]
    rng = np.random.default_rng(sum(map(ord, name + form)))
    c = tsl.coef_init((0.0, 0.0, 0.0), ext, res)
    c.init_value = 0.0126
    n, sd3 = int(c.grid_occ_size), int(c.sub_dim) ** 3
    # blocks within a few metres of the origin, most of them allocated
    b = np.arange(n)
    bx, by = b % int(c.up_dim_x), b // int(c.up_dim_x) % (int(c.up_dim_2) // int(c.up_dim_x))
    alloc = (bx < 5) & (by < 5) & (rng.uniform(size=n) < 0.7)
    alloc[0] = True
    grid = np.where(alloc, (np.cumsum(alloc) - 1) * sd3, -1).astype(np.int32)
    c.data_size = int(alloc.sum()) * sd3
    has = ctypes.c_int(1)
    _lib.check(_lib.lib.tsl_check_class_grid(ctypes.byref(c), _lib.ptr(grid), None, 0, None, ctypes.byref(has)))
    assert has.value == 0
    size = int(c.data_size)
    data = rng.uniform(0.01, 1.0, 300 if form == "palette" else min(size, 500_000)).astype(np.float32)
    data = np.where(rng.uniform(size=size) < 0.5, np.float32(c.init_value), np.resize(data, size)).astype(np.float32)
    ev = tsl.TSDFEvaluator(tsl.CudaSubVoxelMap(c, grid, data=data))
    P, N = 67, 450
    near = np.minimum(np.array(ext), 4.0)
    parts = np.zeros((P, 7), np.float32)
    parts[:, :3] = rng.uniform(-0.2, 1.0, (P, 3)) * near
    parts[:, 3:6] = rng.uniform(-3.1, 3.1, (P, 3))
    parts[:, 6] = 1.0 / P
    parts[5, 0] -= 12.0
    parts[11, 1] -= 40.0
    parts[20, 2] += 2e6
    parts[66, 1] = -3e7
    pts = rng.uniform(-3.0, 3.0, (N, 3)).astype(np.float32)
    tf = np.eye(4, dtype=np.float32)
    tf[:3, 3] = (0.1, -0.2, 0.3)
    return tsl, ev, ob.OracleMap(c, grid, data), parts, pts, np.ascontiguousarray(tf.reshape(-1))


def _alone(tsl, ev, parts, pts, tf, k, pp, chunk, order=0, lookup=0):
    f = tsl.DeviceFilter(ev, parts.shape[0])
    f.set_particles(parts)
    f.set_scan(pts, tf)
    f.set_tile(k, chunk, pp)
    f.set_order(order)
    f.set_block_lookup(lookup)
    s = tsl.Stream()
    f.update_async(s)
    f.sync(s)
    return f.get_particles()[:, 6]


@pytest.mark.parametrize("form", ["palette", "float"])
@pytest.mark.parametrize("name", sorted(MAPS))
def test_values_and_weights(name, form):
    tsl, ev, om, parts, pts, tf = _setup(name, form)
    far = parts.copy()
    far[33, 0] = np.inf
    odd = pts.copy()
    odd[7], odd[100], odd[449], odd[30, 1] = (7e4, 0, 1), (0, -3e38, 0), (np.inf, 1, 1), np.nan
    hits = 0
    for p, q in [(parts, pts), (far, odd)]:
        ref = om.trace(p, q, tf)
        hits += np.count_nonzero(ref < om.coef.data_size)
        assert np.array_equal(ev.trace_indices(p, q, tf), ref)
        got = ev.trace_values(p, q, tf)
        assert np.array_equal(got.view(np.uint32), oracle_values(om, ref).view(np.uint32))
    assert hits > 5000
    for P, N in [(1, 1), (2, 64), (3, 65), (2, 127), (67, 128), (5, 129), (66, 191), (67, 450)]:
        _, w64 = om.evaluate(parts[67 - P:], pts[450 - N:], tf)
        got = ev.evaluate_raw(parts[67 - P:], pts[450 - N:], tf)
        assert np.max(rel_err(got, w64)) <= WEIGHT_RTOL, (P, N)


@pytest.mark.parametrize("form", ["palette", "float"])
@pytest.mark.parametrize("name", sorted(MAPS))
def test_tiles_bit_identical_and_batch_equals_alone(name, form):
    tsl, ev, om, parts, pts, tf = _setup(name, form)
    _, w64 = om.evaluate(parts, pts, tf)
    for chunk in (CHUNK, 0):
        first = None
        for order, lookup in ((0, 0), (1, 0), (0, 1)):
            for k in (1, 2):
                for pp in (1, 2, 4):
                    w = _alone(tsl, ev, parts, pts, tf, k, pp, chunk, order, lookup)
                    key = (chunk, order, lookup, k, pp)
                    assert np.max(rel_err(w, w64 / w64.sum())) <= WEIGHT_RTOL, key
                    first = w if first is None else first
                    assert np.array_equal(w.view(np.uint32), first.view(np.uint32)), key
    members = [(67, 450), (1, 1), (5, 129), (66, 191)]
    filters = []
    for P, N in members:
        f = tsl.DeviceFilter(ev, P)
        f.set_particles(parts[67 - P:])
        f.set_scan(pts[450 - N:], tf)
        filters.append(f)
    b = tsl.Batch(ev, filters)
    s = tsl.Stream()
    for k in (1, 2):
        for pp in (1, 2, 4):
            b.set_tile(k, CHUNK, pp)
            b.update_async(s)
            _, _, status = b.sync(s)
            assert np.all(status == 0)
            for f, (P, N) in zip(filters, members):
                w = _alone(tsl, ev, parts[67 - P:], pts[450 - N:], tf, 1, 1, CHUNK)
                assert np.array_equal(f.get_particles()[:, 6].view(np.uint32), w.view(np.uint32)), (k, pp, P, N)
