"""Kept device blocks: surfaces made on the memory of destroyed ones, one after the other and from two
threads on streams of their own, give the bits of a first surface."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _job(w, stream=None):
    import torch

    from lvr2_amd import HipSurface

    p = torch.from_numpy(w.points).cuda()
    torch.cuda.synchronize()
    s = HipSurface(p, stream=stream)
    s.setKn(w.kn)
    s.setKi(w.ki)
    s.setKd(w.kd)
    s.calculateNormals()
    s.interpolateNormals()
    n = s.getNormals()
    d = s.distances(w.points[::7] + np.float32(1.5), w.voxel)[0]
    idx, d2 = s.kSearch(w.points[::11], 12)
    s.freeGPU()
    return n, d, idx, d2


def _same(a, b):
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)


def test_jobs_on_kept_blocks():
    from lvr2_amd import scenes

    ws = [scenes.plain_small(n, seed) for n, seed in ((20_000, 3), (7_013, 4), (20_000, 5), (33_000, 6))]
    first = [_job(w) for w in ws]
    for _ in range(3):
        for w, want in zip(ws, first):
            _same(_job(w), want)


def test_jobs_of_two_threads():
    import torch

    from lvr2_amd import scenes

    ws = [scenes.plain_small(n, seed) for n, seed in ((20_000, 7), (20_000, 8))]
    want = [_job(w) for w in ws]
    bad = []

    def work(i):
        try:
            st = torch.cuda.Stream()
            with torch.cuda.stream(st):
                for _ in range(5):
                    _same(_job(ws[i], st.cuda_stream), want[i])
        except Exception as e:  # reported by the main thread
            bad.append(e)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad[0]
