"""Destroying a surface while another stream captures: a relaxed capture goes on, and the surface's memory is used
again only when the work on it is done."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RELAXED = 2  # hipStreamCaptureModeRelaxed


def _surface(stream=None):
    import torch

    from lvr2_amd import HipSurface, scenes

    w = scenes.plain_small(5_000)
    s = HipSurface(torch.from_numpy(w.points).cuda(), stream=stream)
    s.setKn(w.kn)
    s.setKi(w.ki)
    s.calculateNormals()
    return s


@pytest.mark.parametrize("own", [False, True])
def test_destroyed_during_a_capture(own):
    import torch

    from lvr2_amd import lib

    hip = lib()  # dlsym finds the runtime's functions through the library
    st, mine = torch.cuda.Stream(), torch.cuda.Stream()
    s = _surface(mine.cuda_stream if own else None)
    x = torch.zeros(256, device="cuda")
    torch.cuda.synchronize()
    assert hip.hipStreamBeginCapture(C.c_void_p(st.cuda_stream), RELAXED) == 0
    with torch.cuda.stream(st):
        x += 1
        s.freeGPU()
        x += 1
    graph = C.c_void_p()
    assert hip.hipStreamEndCapture(C.c_void_p(st.cuda_stream), C.byref(graph)) == 0 and graph
    assert hip.hipGraphDestroy(graph) == 0
    torch.cuda.synchronize()
    assert x.sum().item() == 0  # recorded, not run


def test_moved_surface_is_not_kept():
    """After setStream the former stream may still work on the buffers: they go back to the runtime."""
    import torch

    import lvr2_amd

    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    s = _surface(a.cuda_stream)
    out = torch.empty((5_000, 3), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    lvr2_amd.release_memory()
    s.interpolateNormals()
    s.getNormals(out)
    s.setStream(b.cuda_stream)
    s.freeGPU()
    assert lvr2_amd.release_memory() == 0
    torch.cuda.synchronize()
    want = _surface()
    want.interpolateNormals()
    np.testing.assert_array_equal(out.cpu().numpy(), want.getNormals())
