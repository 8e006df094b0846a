"""The motion update with eight lanes to a particle, at the edges of its
workgroups (32 particles) and of the rule that leaves larger sets to one thread
a particle: within 4e-6 m and 2e-6 rad of the oracle's draws and composition
(the draws' double logarithm, sine and cosine are each side's own)."""
import numpy as np
import pytest

import oracle_binding as ob

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("trig", [0, 2])
@pytest.mark.parametrize("P", [1, 31, 32, 33, 257, 32000, 33000])
def test_motion_sizes(P, trig):
    import tsdf_localization_amd as tsl
    from tsdf_localization_amd import synth
    rng = np.random.default_rng(P)
    parts = np.zeros((P, 7), np.float32)
    parts[:, :3] = rng.uniform(0, 50, (P, 3))
    parts[:, 3:5] = rng.normal(0, 0.3, (P, 2))
    parts[:, 5] = rng.uniform(-np.pi, np.pi, P)
    parts[:, 6] = 1.0 / P
    f = tsl.DeviceFilter(tsl.TSDFEvaluator(synth.room().map, trig=trig), P)
    f.set_particles(parts)
    m = tsl.evaluator.motion_from_delta(0.4, 0.05, 0.01, 0.01, -0.02, 0.15, 0.02, 0.01, seed=99)
    s = tsl.Stream()
    f.motion_async(m, s)
    s.synchronize()
    got = f.get_particles()
    ref = ob.motion(parts, list(m.mean), list(m.stddev), m.seed, trig_mode=ob.trig_mode_for(trig))
    assert np.max(np.abs(got[:, :3] - ref[:, :3])) <= 4e-6
    ang = np.angle(np.exp(1j * (got[:, 3:6].astype(np.float64) - ref[:, 3:6])))
    assert np.max(np.abs(ang)) <= 2e-6
    assert np.array_equal(got[:, 6], ref[:, 6])


@pytest.mark.parametrize("trig", [0, 1, 2])
def test_split_and_single_thread_forms_agree_bit_for_bit(trig):
    """A member's motion does not depend on what else is in its batch: alone
    (eight lanes to a particle) and beside a set of more than 32,768 (one
    thread to a particle) it is the same bits."""
    import tsdf_localization_amd as tsl
    from tsdf_localization_amd import synth
    ev = tsl.TSDFEvaluator(synth.room().map, trig=trig)
    rng = np.random.default_rng(11)
    P = 8191
    parts = np.zeros((P, 7), np.float32)
    parts[:, :3] = rng.uniform(-50, 50, (P, 3))
    parts[:, 3:5] = rng.normal(0, 0.5, (P, 2))
    parts[:, 5] = rng.uniform(-np.pi, np.pi, P)
    parts[:16, 4] = np.float32(np.pi / 2) * rng.choice([-1, 1], 16)  # at the pole
    parts[16:24, 3:6] = 0.0
    parts[:, 6] = 1.0 / P
    m = tsl.evaluator.motion_from_delta(0.4, 0.05, 0.01, 0.01, -0.02, 0.15, 0.02, 0.01, seed=99)
    pts = np.ones((64, 3), np.float32)
    tf = np.ascontiguousarray(np.eye(4, dtype=np.float32).reshape(-1))
    s = tsl.Stream()
    got = []
    for beside in (0, 33000):
        filters = []
        for n in [P] + ([beside] if beside else []):
            f = tsl.DeviceFilter(ev, n)
            f.set_particles(np.resize(parts, (n, 7)))
            f.set_scan(pts, tf)
            filters.append(f)
        b = tsl.Batch(ev, filters)
        b.motion_async([m] * len(filters), s)
        b.sync(s)
        got.append(filters[0].get_particles())
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
    assert not np.array_equal(got[0][:, :6], parts[:, :6])
