"""The vertex moves of the planar marching cubes where both best-first passes give up: the tile kernel then finds
a vertex's neighbours, and the vertex's next move must start from what that search found."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NEAR = [(0, 0, 0), (40, 10, 0), (10, 50, 5), (60, 60, 10), (200, 180, 90)]


def _position(code):
    """The point whose 63-bit Morton code (x highest) is code, in a frame of cells of size 1."""
    return tuple(sum(((code >> (3 * b + 2 - a)) & 1) << b for b in range(21)) for a in range(3))


def _deep_cloud():
    """118,800 points whose tree is 64 chains of 57 levels side by side.  From far away (all distances equal in
    fp32) a query sees every leaf within its bound: the lane search's pool overflows after 137 leaves, and
    the wave search, which goes down the 64 chains at once, leaves 192 entries behind at every second
    level: 5,632 at the most, of the 4,096 that its stack holds."""
    p = NEAR + [(5000, 5000, 5000)] * 11
    for c in range(64):
        for j in range(58):
            rest = 57 - j
            code = (c << 57) | (((1 << j) - 1) << rest) | (((1 << (rest - 1)) - 1) if j < 57 else 0)
            p += [_position(code)] * 32
    return np.array(p, np.float32)


def test_moves_after_a_search_that_outgrew_the_best_first_passes():
    import torch

    from lvr2_amd import HipSurface

    p = _deep_cloud()
    assert p.min() == 0.0 and p.max() == 2097151.0
    V = 2.0 ** 48
    s = HipSurface(p)
    v, _, _ = s.grid(V, extrude=True, box=(-1.5 * V, -2.5 * V, -2.5 * V, 1.5 * V, 2.5 * V, 2.5 * V))
    # the surface x = V / 2, kept in four cells with two border edges each: the eight border vertices move twice
    dist = torch.from_numpy((v[:, 0] - V / 2).astype(np.float32)).cuda()
    gone = torch.from_numpy(((v[:, 1] < -V / 2) | (v[:, 2] < -V / 2)).astype(np.uint8)).cuda()
    start, faces = s.mesh(dist, gone, "MC")
    border = (start[:, 1:] != V).any(1)
    assert len(faces) == 8 and border.sum() == 8
    s.setProfiling(True)
    got, _ = s.mesh(dist, gone, "PMC")
    # every border vertex was left by both passes of its first search (the tile kernel counts here too)
    assert s.kernelStats()["other"]["refine"] >= 16
    # first move: all points are equally far, the first five win; second move: they are the nearest
    want = np.array(NEAR, np.float64).mean(0)
    np.testing.assert_allclose(got[border], np.broadcast_to(want, (8, 3)), rtol=1e-6)
    np.testing.assert_array_equal(got[~border], start[~border])
