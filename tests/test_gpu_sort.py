"""Clouds and lattices on both sides of the lines where the radix sort changes its form (1,024-key tiles up to
1,048,576 keys, 4,096-key tiles, the table scan above 4,194,304 keys; an odd or even number of passes): a
wrong order would lose points from the leaves, so searches are compared with the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 1_023, 1_024, 1_025, 16_385, 1_048_576, 1_048_577, 4_194_304, 4_194_305])
def test_build_sizes(oracle_mod, n):
    from lvr2_amd import HipSurface, scenes

    p = scenes.sphere_torus(11, n, 1.0, 0.01)
    s = HipSurface(p)
    o = oracle_mod.Surface(p)
    rng = np.random.default_rng(1)
    q = np.concatenate([p[rng.integers(0, n, 150)], p[:2], p[-2:]])
    k = min(n, 9)
    gi, gd = s.kSearch(q, k)
    oi, od = o.knn(q, k)
    np.testing.assert_array_equal(gi, oi)
    np.testing.assert_array_equal(gd, od)


@pytest.mark.parametrize("nscans", [2, 256, 257])
def test_scan_counts(oracle_mod, nscans):
    from lvr2_amd import HipSurface, scenes

    p = scenes.plane_boxes_sphere(5, 70 * nscans, 0.5)
    s = HipSurface(p, scan_sizes=[70] * nscans)
    s.setKn(2)
    s.setKi(0)
    s.calculateNormals()
    k = s.adaptiveK()
    for i in {0, 1, nscans // 2, nscans - 1}:
        want = oracle_mod.Surface(p[70 * i:70 * (i + 1)]).normals(2, 3, (1e6, 1e6, 1e6))[2]
        np.testing.assert_array_equal(k[70 * i:70 * (i + 1)], want)


@pytest.mark.parametrize("shift,voxel", [((0.0, 0.0, 0.0), 10.0), ((5e4, -8e4, 3e3), 10.0), ((0.0, 0.0, 0.0), 3.1),
                                         ((-700.0, 0.0, 900.0), 60.0)])
def test_lattice_offsets(oracle_mod, shift, voxel):
    """The lattice keys are relative to the box: far from the origin, and with other key widths."""
    from lvr2_amd import HipSurface, scenes

    p = (scenes.plane_boxes_sphere(6, 20_000, 0.5) + np.asarray(shift, np.float32)).astype(np.float32)
    v, c, ci = HipSurface(p).grid(voxel)
    ov, oc, oci = oracle_mod.grid(p, oracle_mod.Surface(p).bbox(), voxel, extrude=True)
    np.testing.assert_array_equal(ci, oci)
    np.testing.assert_array_equal(c, oc)
    np.testing.assert_array_equal(v, ov)


@pytest.mark.parametrize("sizes", [[4_096, 65, 64, 4_095, 9_000], [64] * 70 + [5_000], [4_200_000, 70, 300_000],
                                   [66, 4_300_000]])
def test_scan_boxes(oracle_mod, sizes):
    """Scan bounds inside, at the ends of and across the blocks and rows the scan boxes are reduced in."""
    from lvr2_amd import HipSurface, scenes

    p = scenes.plane_boxes_sphere(7, sum(sizes), 0.5)
    s = HipSurface(p, scan_sizes=sizes)
    s.setKn(2)
    s.setKi(0)
    s.calculateNormals()
    k = s.adaptiveK()
    off = np.concatenate([[0], np.cumsum(sizes)])
    for i in {0, 1, len(sizes) - 2, len(sizes) - 1}:
        a = p[off[i]:off[i + 1]]
        if len(a) <= 10_000:
            want = oracle_mod.Surface(a).normals(2, 3, (1e6, 1e6, 1e6))[2]
        else:
            one = HipSurface(a)
            one.setKn(2)
            one.setKi(0)
            one.calculateNormals()
            want = one.adaptiveK()
        np.testing.assert_array_equal(k[off[i]:off[i + 1]], want)
