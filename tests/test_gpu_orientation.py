"""The orientation of normals seen edge-on.

A scanner's range noise lies along its rays, so every point of a wall whose plane runs through the scanner
stays in that plane: n . (f - q) is zero up to rounding, and the order in which a neighbourhood's moments
are added up decides the normal's sign.  The interpolation adds neighbours' normals, so one reversed normal can
reverse others beside it.  The k-set does not fix these signs; what fixes them is that the search tries the
same radii in the same order, launch after launch and build after build.  The signs recorded in
golden/orientation_golden.npz are those of the rounds searched one after the other (written by
`python tests/test_gpu_orientation.py`, which runs the searches and saves what they give).
"""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PATH = os.path.join(ROOT, "tests", "golden", "orientation_golden.npz")
SCANNER = np.array([0.0, 0.0, 1.75])
# horizontal directions of the walls, exact in fp64 up to one rounding (no trigonometry: the same cloud everywhere)
DIRS = [(3 / 5, 4 / 5), (-5 / 13, 12 / 13), (-15 / 17, -8 / 17), (20 / 29, -21 / 29), (999 / 1000.9, 60 / 1000.9),
        (-40 / 1600.5, 1600 / 1600.5)]
CASES = [("small", 6_000, 10, 10), ("odd", 40_013, 20, 10), ("wide", 120_000, 50, 20), ("runs", 700_000, 10, 10)]


def cloud(n):
    """n points on the walls, in rays from the scanner with noise along the ray, and which wall each is on."""
    rng = np.random.default_rng(n)
    w = np.sort(rng.integers(0, len(DIRS), n))
    d = np.array(DIRS)[w]
    r = 5.0 + 20.0 * rng.random(n)
    up = rng.random(n) * 0.4 - 0.07  # tangent of the elevation
    r = r + 0.003 * (rng.random(n) - 0.5)
    p = np.stack([r * d[:, 0], r * d[:, 1], SCANNER[2] + r * up], 1)
    return p.astype(np.float32), w


def signs(n, kn, ki):
    """Of up to about 50,000 points: on their wall's left-hand side, normals and interpolated normals, and edge-on."""
    from lvr2_amd import HipSurface

    p, w = cloud(n)
    s = HipSurface(p)
    s.setKn(kn)
    s.setKi(ki)
    s.setFlippoint(*SCANNER)
    s.calculateNormals()
    raw = s.getNormals().astype(np.float64)
    s.interpolateNormals()
    left = np.array([(-y, x, 0.0) for x, y in DIRS])[w]
    to = SCANNER - p
    edge = np.abs((raw * to).sum(1)) < 1e-5 * np.linalg.norm(to, axis=1)
    some = slice(None, None, max(1, n // 50_000))
    return (raw * left).sum(1)[some] > 0, (s.getNormals() * left).sum(1)[some] > 0, edge[some]


@pytest.mark.gpu
@pytest.mark.parametrize("name,n,kn,ki", CASES)
def test_signs_of_edge_on_normals(name, n, kn, ki):
    want = np.load(PATH)
    raw, interp, edge = signs(n, kn, ki)
    assert edge.mean() > 0.9 and 0.1 < raw.mean() < 0.9  # the signs are open, and both occur
    assert int((raw != np.unpackbits(want[f"{name}_raw"], count=len(raw)).astype(bool)).sum()) == 0
    assert int((interp != np.unpackbits(want[f"{name}_interpolated"], count=len(raw)).astype(bool)).sum()) == 0


if __name__ == "__main__":
    out = {}
    for name_, n_, kn_, ki_ in CASES:
        a, b, e = signs(n_, kn_, ki_)
        out[f"{name_}_raw"], out[f"{name_}_interpolated"] = np.packbits(a), np.packbits(b)
        print(name_, n_, "edge-on", e.mean(), "left", a.mean(), b.mean())
    np.savez_compressed(sys.argv[1] if len(sys.argv) > 1 else PATH, **out)
