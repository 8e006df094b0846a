"""Resampling in one workgroup, at the edges of its two sizes (2048 and 8192
candidates) and past them: source indices and particles of the oracle's
sequential draw."""
import numpy as np
import pytest

import oracle_binding as ob

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["even", "uneven", "sparse"])
@pytest.mark.parametrize("M", [1, 1023, 2045, 2046, 2047, 2049, 5000, 8189, 8190, 8191, 8193])
def test_resample_sizes(M, kind):
    import tsdf_localization_amd as tsl
    rng = np.random.default_rng(M)
    w = np.ones(M) if kind == "even" else rng.gamma(0.5 if kind == "uneven" else 0.01, size=M) + 1e-12
    parts = np.zeros((M, 7), np.float32)
    parts[:, 0] = np.arange(M)
    parts[:, 6] = (w / w.sum()).astype(np.float32)
    for u0 in (0.0, 0.37 / M, 0.999 / M):
        new, idx = tsl.resample_systematic(parts, np.float32(u0))
        ref = ob.resample(parts[:, 6], np.float32(u0))
        assert np.array_equal(idx, ref)
        assert np.array_equal(new, parts[ref])


@pytest.mark.parametrize("M", [6000, 6135, 6140, 6142, 6143, 6144, 6145, 6160])
def test_resample_sizes_at_the_larger_workgroups_edge(M):
    import tsdf_localization_amd as tsl
    rng = np.random.default_rng(M)
    for shape in (4.0, 0.01):
        w = rng.gamma(shape, size=M) + 1e-12
        parts = np.zeros((M, 7), np.float32)
        parts[:, 0] = np.arange(M)
        parts[:, 6] = (w / w.sum()).astype(np.float32)
        for u0 in (0.0, 0.37 / M, 0.999 / M):
            new, idx = tsl.resample_systematic(parts, np.float32(u0))
            ref = ob.resample(parts[:, 6], np.float32(u0))
            assert np.array_equal(idx, ref)
            assert np.array_equal(new, parts[ref])
