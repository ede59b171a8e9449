"""Device memory kept between calls goes back to the runtime: when asked, and when later calls leave it alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _free():
    import torch

    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_release_after_the_last_surface():
    import lvr2_amd
    from lvr2_amd import HipSurface, scenes

    lvr2_amd.release_memory()
    w = scenes.plain_small(400_000)
    s = HipSurface(w.points)
    s.setKn(10)
    s.calculateNormals()
    del s
    before = _free()
    got = lvr2_amd.release_memory()
    assert got > 400_000 * 36  # its moments alone
    assert _free() - before >= got // 2  # the runtime frees in pages of its own
    assert lvr2_amd.release_memory(0) == 0
    s = HipSurface(w.points)  # and the next one works
    assert s.kSearch(w.points[:7], 1)[0][:, 0].tolist() == list(range(7))


def test_host_calls_age_what_they_do_not_use():
    import lvr2_amd
    from lvr2_amd import HipSurface, scenes

    p = scenes.plain_small(20_000).points
    s = HipSurface(p)
    lvr2_amd.release_memory()
    s.kSearch(np.tile(p, (50, 1)), 8)  # buffers of 76 MB, kept
    for _ in range(100):
        s.kSearch(p[:10], 8)
    assert lvr2_amd.release_memory() < 1 << 20
