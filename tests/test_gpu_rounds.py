"""The adaptive rounds out of order: the neighbourhood size every point stops at, and how many points
reach each round, bit-exact against the oracle's round-by-round loop, on both sides of the lines where the
order of the searches changes (all rounds at once up to 16,384 rejected points and a quarter of the cloud;
round 5 first only where at most 45 % of the points are rejected), single- and multi-scan, and against the merged rounds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _cloud(scene, n):
    from lvr2_amd import scenes

    if scene == "plain":
        return scenes.plain_small(n), (0.0, 0.0, 0.0)
    if scene == "outdoor":
        p, sc = scenes.outdoor_scan(3, n)
        return scenes.Workload("outdoor", p, 50, 20, 10, tuple(float(c) for c in sc), 0.2), tuple(map(float, sc))
    n_el = max(4, int(round(np.sqrt(n / 2.56))))
    return scenes.room(-(-n // n_el), n_el), (0.0, 0.0, 0.0)


def _stats(k, kn):
    """Points whose search reaches round r: those that do not stop at a smaller k (32 kn <= n)."""
    return [int(np.sum(k >= kn << r)) for r in range(1, 6)]


@pytest.mark.parametrize("scene,n,kn,few", [
    ("plain", 700, 10, True),       # k clamped to the cloud in round 5 and below
    ("plain", 3_001, 10, True),
    ("plain", 30_000, 10, True),
    ("outdoor", 20_011, 10, None),
    ("outdoor", 60_007, 20, False),  # most points rejected: round 3 first
    ("room", 90_000, 20, False),     # about a quarter rejected: round 5 first
])
def test_adaptive_k_and_counts(oracle_mod, scene, n, kn, few):
    from lvr2_amd import HipSurface

    w, flip = _cloud(scene, n)
    o = oracle_mod.Surface(w.points)
    want = o.normals(kn, 3, flip)[2]
    s = HipSurface(w.points)
    s.setKn(kn)
    s.setKi(10)
    s.setFlippoint(*flip)
    s.calculateNormals()
    np.testing.assert_array_equal(s.adaptiveK(), want)
    st = s.normalsStats()
    if few is not None:
        assert (st[1] <= 16_384) == few
    if len(w.points) >= 32 * kn:
        assert st.tolist() == _stats(want, kn)
    normals = s.getNormals()
    assert np.all(np.isfinite(normals))
    s.setRetryMode(True)
    s.calculateNormals()
    np.testing.assert_array_equal(s.adaptiveK(), want)


def test_adaptive_k_of_scans(oracle_mod):
    """Two scans of different density in one handle: each point's k equals its own scan's."""
    from lvr2_amd import HipSurface

    a, _ = _cloud("plain", 9_000)
    b, _ = _cloud("room", 40_000)
    s = HipSurface(np.concatenate([a.points, b.points]), scan_sizes=[len(a.points), len(b.points)])
    s.setKn(10)
    s.setKi(10)
    s.calculateNormals()
    want = np.concatenate([oracle_mod.Surface(w.points).normals(10, 3, (1e6, 1e6, 1e6))[2] for w in (a, b)])
    np.testing.assert_array_equal(s.adaptiveK(), want)


@pytest.mark.parametrize("lone", [1, 7, 44, 101])
def test_lone_patches_beside_a_dense_one(oracle_mod, lone):
    """Patches of fewer points than k, whose searches reach a dense patch just as their radius does."""
    from lvr2_amd import HipSurface

    rng = np.random.default_rng(lone)
    flat = np.array([1.0, 1.0, 0.02])
    dense = rng.uniform(-2, 2, (12_000, 3)) * flat
    far = [rng.uniform(-0.1, 0.1, (lone, 3)) * flat + np.array([d, 0.3 * d, 0.0]) for d in (6.0, -33.0, 80.0)]
    p = np.concatenate([dense] + far).astype(np.float32)
    s = HipSurface(p)
    s.setKn(50)
    s.setKi(20)
    s.calculateNormals()
    np.testing.assert_array_equal(s.adaptiveK(), oracle_mod.Surface(p).normals(50, 3, (1e6, 1e6, 1e6))[2])
