"""Profiling with and without the work counters: timers either way, the same results."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counters", [False, True])
def test_counters_are_optional(counters):
    from lvr2_amd import HipSurface, scenes

    w = scenes.plain_small(30_000)
    s = HipSurface(w.points)
    s.setKn(w.kn)
    s.setKi(w.ki)
    s.setKd(w.kd)

    def run():
        s.calculateNormals()
        n = s.getNormals()
        return n, s.distances(w.points[::9] + np.float32(1.0), w.voxel)[0]

    want = run()
    s.setProfiling(True, counters=counters)
    got = run()
    for a, b in zip(want, got):
        np.testing.assert_array_equal(a, b)
    ms, launches = s.timings()["normals_first"]
    assert launches == 1 and ms > 0
    st = s.kernelStats()
    assert (st["round1"]["tiles"] > 0) == counters and (st["sdf"]["resolved"] > 0) == counters
