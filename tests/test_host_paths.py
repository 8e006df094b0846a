"""Host paths of the library that need a device to run, on the CPU: libtsl.so
over the stand-in of the HIP runtime in cpp/hip_stub.cpp (device memory is host
memory, kernels do nothing, asynchronous copies run when something waits for
them).  Each test runs in a process of its own."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # before libtsl.so
stub.stub_live_bytes.restype = ctypes.c_size_t
stub.stub_set_total.argtypes = [ctypes.c_size_t]
stub.stub_fail_launch.argtypes = stub.stub_fail_copy.argtypes = [ctypes.c_long]
import numpy as np
import tsdf_localization_amd as tsl

def host_map(ext=(3.0, 3.0, 2.0), res=0.05):
    c = tsl.coef_init((0, 0, 0), ext, res, 0.25)
    n = int(c.grid_occ_size)
    sd3 = int(c.sub_dim) ** 3
    c.data_size = n * sd3
    grid = (np.arange(n) * sd3).astype(np.int32)
    return tsl.CudaSubVoxelMap(c, grid, data=np.resize(np.float32([0.5, 0.75]), n * sd3))
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    out = tmp_path_factory.mktemp("stub") / "libhipstub.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-Wall", "-I", "/opt/rocm/include", "-o", str(out),
                    os.path.join(HERE, "cpp", "hip_stub.cpp")], check=True)
    return out


def run(stub, code):
    r = subprocess.run([sys.executable, "-c", PRELUDE + code, str(stub)], cwd=os.path.dirname(HERE),
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


@pytest.mark.parametrize("ext,res", [((3.0, 3.0, 2.0), 0.05), ((3.0, 3.0, 2.0), 0.04)])
def test_map_bytes_and_server_budget_hold_the_class_grid(stub, ext, res):
    """tsl_map_device_bytes is what the map holds on the device, with a class
    grid (0.05 m) and without (0.04 m), and a server's budget starts from it."""
    out = run(stub, f"""
from tsdf_localization_amd.server import Server
m = host_map({ext}, {res})
before = stub.stub_live_bytes()
d = m.device_map()
held = stub.stub_live_bytes() - before
print("voxels", 2 * m.dataSize(), "held", held)
assert d.device_bytes() == held, (d.device_bytes(), held)
s = Server(tsl.TSDFEvaluator(m), max_robots=2, max_particles=100)
assert s.stats()["used_bytes"] == held
s.close()
""")
    print(out)


def test_class_grid_leaves_the_device_room(stub):
    """A class grid takes no more than an eighth of the free memory: with less
    free, the map is loaded without one and filters keep the room."""
    run(stub, """
m = host_map()
full = m.device_map().device_bytes()
grid = full - 2 * m.dataSize()
for times in (4, 12):  # what is free once the voxels are loaded, in class grids
    m = host_map()
    stub.stub_set_total(stub.stub_live_bytes() + 2 * m.dataSize() + times * grid)
    d = m.device_map()
    assert (d.device_bytes() == full) == (times == 12), (times, d.device_bytes(), full)
    tsl.DeviceFilter(tsl.TSDFEvaluator(m), int(0.85 * times * grid) // 120)  # 116 bytes a particle
""")


@pytest.mark.parametrize("call", ["evaluate", "evaluate_cloud", "set_scan", "set_scan_raw"])
@pytest.mark.parametrize("step", ["launch", "copy"])
def test_failed_call_leaves_no_copy_of_the_callers_arrays(stub, call, step):
    """Whichever launch or copy of a call fails, when it returns no queued copy
    reads or writes the caller's arrays (large enough not to be staged)."""
    run(stub, f"""
ev = tsl.TSDFEvaluator(host_map())
f = tsl.DeviceFilter(ev, 16)
pts = np.ones((30000, 3), np.float32)
rings = np.zeros(30000, np.int16)
parts = np.ones((20000, 7), np.float32)
tf = np.eye(4, dtype=np.float32)
calls = dict(evaluate=lambda: ev.evaluate(parts, pts, tf), evaluate_cloud=lambda: ev.evaluate_cloud(parts, pts, rings, tf),
             set_scan=lambda: f.set_scan(pts, tf), set_scan_raw=lambda: f.set_scan_raw(pts, rings, tf, 0.064))
fail = stub.stub_fail_{step}
for after in range(100):
    fail(after)
    try:
        calls["{call}"]()
        fail(-1)
        break
    except RuntimeError:
        assert stub.stub_pending() == 0, after
assert 0 < after < 100
assert stub.stub_pending() == 0
""")


def test_call_out_of_memory_leaves_no_copy_of_the_callers_arrays(stub):
    """The same where the particles find no device memory after the scan has
    been queued."""
    run(stub, """
ev = tsl.TSDFEvaluator(host_map())
ev.evaluate(np.ones((16, 7), np.float32), np.ones((30000, 3), np.float32), np.eye(4, dtype=np.float32))
stub.stub_set_total(stub.stub_live_bytes())
try:
    ev.evaluate(np.ones((20000, 7), np.float32), np.ones((30000, 3), np.float32), np.eye(4, dtype=np.float32))
    raise SystemExit("did not fail")
except RuntimeError:
    assert stub.stub_pending() == 0
""")


def test_scan_setters_without_pinned_staging(stub):
    """A filter whose staging finds no pinned memory copies without it."""
    run(stub, """
f = tsl.DeviceFilter(tsl.TSDFEvaluator(host_map()), 16)
stub.stub_no_pinned(1)
tf = np.eye(4, dtype=np.float32)
f.set_scan(np.ones((100, 3), np.float32), tf)
f.set_scan_raw(np.ones((100, 3), np.float32), np.zeros(100, np.int16), tf, 0.064)
f.get_particles()
""")


def test_wide_map_evaluates_as_many_items_as_with_two_particles(stub):
    """The 64-bit form's automatic tile (one particle per wavefront) refuses no
    particles x chunks that two per wavefront can launch."""
    run(stub, """
c = tsl.coef_init((0, 0, 0), (3.0, 3.0, 2.0), 0.05, 0.25)
n, sd3 = int(c.grid_occ_size), int(c.sub_dim) ** 3
c.data_size = n * sd3
m = tsl.CudaSubVoxelMap(c, np.arange(n, dtype=np.int64) * sd3, tsdf_mm=np.zeros(n * sd3, np.int16), truncation_mm=300,
                        sigma=0.1)
P, N = 230_000, 64 * 40_000
f = tsl.DeviceFilter(tsl.TSDFEvaluator(m), P)
f.set_particles(np.ones((P, 7), np.float32))
f.set_scan(np.ones((N, 3), np.float32), np.eye(4, dtype=np.float32))
assert 2 ** 31 < (P + 3) // 4 * (N // 64) < 2 ** 32
f.set_tile(0, 64, 0)
f.update_async()
""")


@pytest.mark.parametrize("res,filter_shapes,batch_shapes", [(0.05, 6, 4), (0.04, 60, 24)])
def test_autotuners_time_each_distinct_shape_once(stub, res, filter_shapes, batch_shapes):
    """On a class grid (0.05 m) neither K nor points per lane shapes the kernel:
    what differs are the chunks (five lengths, the automatic one by K; a
    batch's four).  Without one (0.04 m): two lookups x six shapes x five
    lengths, a batch's six shapes x four.  Each in both particle orders, whose
    own time is measured too."""
    run(stub, f"""
ev = tsl.TSDFEvaluator(host_map(res={res}))
f = tsl.DeviceFilter(ev, 64)
f.set_particles(np.ones((64, 7), np.float32))
f.set_scan(np.ones((5000, 3), np.float32), np.eye(4, dtype=np.float32))
stub.stub_timings()
f.autotune(reps=1)
assert stub.stub_timings() == 2 * (1 + {filter_shapes})
b = tsl.Batch(ev, [f])
b.set_tile(1, 0, 4)
k, pp, chunk, ms = b.autotune(tsl.Stream(), reps=1)
assert stub.stub_timings() == {batch_shapes}
""")


def test_spatial_order_of_the_allocation_free_entry(stub):
    """The order's launches come only where there are pairs enough to pay for
    them: not for short scans, nor for few pairs."""
    run(stub, """
ev = tsl.TSDFEvaluator(host_map())
tf = np.eye(4, dtype=np.float32)
tf_p = ctypes.c_void_p(tf.ctypes.data)
def launches(P, N):
    p, q, w = np.ones((P, 7), np.float32), np.ones((N, 3), np.float32), np.empty(P, np.float32)
    stub.stub_launches()
    rc = tsl._lib.lib.tsl_evaluate_raw_noalloc(ev.handle, tsl._lib.ptr(p), P, tsl._lib.ptr(q), N, tf_p,
                                               tsl._lib.ptr(w), None)
    assert rc == 0
    return stub.stub_launches()
plain = launches(1000, 300)
for P, N, ordered in [(8191, 5000, False), (8192, 4095, False), (8192, 4096, True), (20000, 64, False),
                      (200000, 255, False), (200000, 256, True), (100000, 335, False), (100000, 336, True)]:
    assert (launches(P, N) > plain) == ordered, (P, N)
""")


def test_lone_filters_resample_in_one_launch_up_to_6144_candidates(stub):
    run(stub, """
ev = tsl.TSDFEvaluator(host_map())
for n, one in [(2000, True), (2100, True), (6100, True), (6200, False), (8100, False)]:
    f = tsl.DeviceFilter(ev, n)
    f.set_particles(np.ones((n, 7), np.float32))
    stub.stub_launches()
    f.resample_async(np.float32(0.3 / n))
    first = stub.stub_launches()
    f.resample_async(np.float32(0.3 / n))
    assert (stub.stub_launches() == 1) == one, (n, first)
""")
