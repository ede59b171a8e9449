"""Which search a batch of queries takes: up to 1,024 every query gets a wave of its own, so that a query with
hundreds of leaves at almost one distance does not wait for a single lane; either way the oracle's neighbours."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ball(oracle_mod):
    from lvr2_amd import HipSurface

    p = np.random.default_rng(1).normal(size=(30_000, 3))
    p = (p / np.linalg.norm(p, axis=1, keepdims=True)).astype(np.float32)
    return HipSurface(p), oracle_mod.Surface(p)


@pytest.mark.parametrize("m,lanes", [(1, False), (1_024, False), (1_025, True)])
@pytest.mark.parametrize("scale", [0.5, 20.0])
def test_route(ball, m, lanes, scale):
    s, o = ball
    q = (np.random.default_rng(m).normal(size=(m, 3)) * scale).astype(np.float32)
    s.setProfiling(True)
    s.kernelStats(reset=True)
    gi, gd = s.kSearch(q, 10)
    st = s.kernelStats(reset=True)["other"]
    s.setProfiling(False)
    # the lane search counts its slowest lanes' leaves; the wave search has no such count
    assert (st["attempts"] > 0) == lanes
    assert st["resolved"] == m
    oi, od = o.knn(q, 10)
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gd, od)
