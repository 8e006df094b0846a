"""The order of a prepared scan: by the Morton code of its 0.25 m cells, ties
in the caller's order, at the edges of the sort's tiles, of its staged rounds
and of the rule that leaves long scans to the radix sort.  Two filters get the
same points, one of them already in that order, which a stable sort leaves as
it is: every weight must be the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _morton(pts):
    c = np.clip(np.floor(pts * np.float32(4)) + np.float32(1048576), 0, 2097151)
    c = np.where(np.isnan(pts), 0, c).astype(np.uint64)
    key = np.zeros(len(pts), np.uint64)
    for b in range(21):
        for a in range(3):
            key |= ((c[:, a] >> np.uint64(b)) & np.uint64(1)) << np.uint64(3 * b + a)
    return key


@pytest.mark.parametrize("n", [1, 2, 63, 255, 256, 257, 511, 513, 2049, 8192, 8193, 16641, 65536, 65537])
def test_scan_order(n):
    import tsdf_localization_amd as tsl
    from tsdf_localization_amd import synth
    room = synth.room()
    ev = tsl.TSDFEvaluator(room.map)
    rng = np.random.default_rng(n)
    pts = rng.uniform(-4, 4, (n, 3)).astype(np.float32)
    pts[: n // 3] = pts[0]  # one cell for many
    if n > 300:
        pts[5], pts[290] = (3e5, -3e5, 1e30), (np.inf, -np.inf, 0)
    order = np.argsort(_morton(pts), kind="stable")
    weights = []
    for q in (pts, pts[order]):
        f = tsl.DeviceFilter(ev, 64)
        f.set_particles(room.particles[:64])
        f.set_scan(q, room.tf)
        s = tsl.Stream()
        f.update_async(s)
        f.sync(s)
        weights.append(f.get_particles()[:, 6])
    assert np.array_equal(weights[0].view(np.uint32), weights[1].view(np.uint32))
