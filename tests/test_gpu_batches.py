"""Best-first searches of few and many queries (the batch size sets how many lanes of a wave search: 1 to
64) against the oracle, on a cloud with repeated points, from each output that the search feeds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def surface(oracle_mod):
    from lvr2_amd import HipSurface, scenes

    p = scenes.sphere_torus(21, 40_000, 1.0, 0.01)
    p[30_000:] = p[:10_000]  # every key of these has a tie
    n = (-p / np.linalg.norm(p, axis=1, keepdims=True)).astype(np.float32)
    s = HipSurface(p)
    s.setNormals(n)
    return s, oracle_mod.Surface(p), p, n


@pytest.mark.parametrize("m", [1, 2, 63, 64, 65, 767, 769, 3_073, 12_289, 49_151, 49_153])
@pytest.mark.parametrize("k", [5, 10, 16, 17, 32])
def test_batch_sizes(surface, m, k):
    from lvr2_amd import scenes

    s, o, p, n = surface
    q = scenes.band_queries(p, m, 0.2, m + k)
    gi, gd = s.kSearch(q, k)
    oi, od = o.knn(q, k)
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gd, od)
    s.setKd(k)
    proj, eucl, _ = s.distances(q, 0.05)
    op, oe = o.distance(n, k, q)
    np.testing.assert_array_equal(proj, op)
    np.testing.assert_array_equal(eucl, oe)
