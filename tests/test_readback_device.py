"""Positions into device memory, which only the runtime may copy to, on both sides of the pinned
staging limit and before and after calls with host destinations."""
import ctypes

import numpy as np
import pytest

from ckmpm_amd import native
from tests.test_readback import _engine


@pytest.mark.gpu
@pytest.mark.parametrize("side", [3, 22, 23])  # 213, 85k and 97k particles; 87,381 fit the staging
@pytest.mark.parametrize("host_first", [False, True])
def test_positions_into_device_memory(side, host_first):
    import torch

    e = _engine(side)
    for k in range(2):
        e.Substep(0.0 if k == 0 else 1e-4, 1e-4)
    n = e.n(0)
    want = e.positions(0) if host_first else None
    lib = native.load()
    for shift in (0, 1, 5):
        buf = torch.full((3 * n + 16,), -7.0, device="cuda")
        torch.cuda.synchronize()
        p = ctypes.cast(buf.data_ptr() + 4 * shift, ctypes.POINTER(ctypes.c_float))
        cnt = ctypes.c_uint64()
        assert lib.ckmpm_get_positions(e._h, 0, p, n, ctypes.byref(cnt)) == native.OK and cnt.value == n
        got = buf.cpu().numpy()
        if want is None:
            want = e.positions(0)
        np.testing.assert_array_equal(got[shift:shift + 3 * n].reshape(n, 3), want)
        assert (got[:shift] == -7).all() and (got[shift + 3 * n:] == -7).all()
        np.testing.assert_array_equal(e.positions(0), want)
    e.close()
