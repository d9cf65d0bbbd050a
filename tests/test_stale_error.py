"""An error that another HIP call of the thread has left behind is not the engine's: reads of
its status and positions succeed all the same, and leave the error to whoever asks for it."""
import ctypes

import numpy as np
import pytest

from ckmpm_amd import native, scenes
from ckmpm_amd.engine import engine_from_scene


def _leave_error(lib):
    assert lib.hipSetDevice(1 << 20) != 0  # no such device: refused by the runtime


@pytest.mark.gpu
def test_reads_do_not_report_an_earlier_error():
    import torch

    torch.cuda.init()
    lib = native.load()
    sc = scenes.colliding_spheres()
    lib.hipGetLastError()
    _leave_error(lib)
    kept = lib.hipPeekAtLastError() != 0  # a runtime may drop it with the next good call
    e = engine_from_scene(sc)             # sets up, which reads the status
    want = e.positions(0)
    for dest in (np.zeros((e.n(0), 3), np.float32), torch.zeros((e.n(0), 3), pin_memory=True).numpy()):
        lib.hipGetLastError()
        _leave_error(lib)
        e.Synchronize()
        assert e.counters().flags == 0
        cnt = ctypes.c_uint64()
        p = dest.ctypes.data_as(ctypes.POINTER(ctypes.c_float))
        assert lib.ckmpm_get_positions(e._h, 0, p, e.n(0), ctypes.byref(cnt)) == native.OK
        np.testing.assert_array_equal(dest, want)
        if kept:
            assert lib.hipPeekAtLastError() != 0
    lib.hipGetLastError()
    e.close()
