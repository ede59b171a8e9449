"""Lists of more than 1,024 blocks of 4,096 entries: their compaction scans the block counts in a launch of its own
instead of summing them in every block.  A project of that size against its scans one by one, whose lists are
short, on both sides of the line."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIRST = 2_000_003
LINE = 1024 * 4096


def _run(p, sizes=None):
    from lvr2_amd import HipSurface

    s = HipSurface(p, scan_sizes=sizes)
    s.setKn(10)
    s.setKi(10)
    s.calculateNormals()
    return s.adaptiveK(), s.normalsStats(), s.getNormals()


@pytest.mark.parametrize("n", [LINE, LINE + 1, LINE + 300_001])
def test_rounds_above_the_line(n):
    from lvr2_amd import scenes

    a = scenes.room_scan(3, 2_000, 1_001)[:FIRST]
    b, _ = scenes.outdoor_scan(3, n - FIRST)
    ka, sa, na = _run(a)
    kb, sb, nb = _run(b)
    k, st, nn = _run(np.concatenate([a, b]), [len(a), len(b)])
    np.testing.assert_array_equal(k, np.concatenate([ka, kb]))
    np.testing.assert_array_equal(st, sa + sb)
    assert st[1] > 100_000  # each round has a list
    assert st[4] > 10_000
    want = np.concatenate([na, nb]).astype(np.float64)
    # a flat neighbourhood's normal is good to the rounding of its moments; its sign is not compared
    c = np.abs((want * nn).sum(1))
    assert np.quantile(c, 1e-3) > 1 - 1e-6 and (c > 0.99).mean() > 0.9999
