"""Positions into every kind of destination: pageable and pinned memory, offset into a pinned
allocation, at sizes on both sides of the pinned staging limit, with guard words around the
destination; and the status the host reads."""
import ctypes

import numpy as np
import pytest

from ckmpm_amd import native, scenes
from ckmpm_amd.engine import engine_from_scene


def _engine(side, offset=0.0):
    r = np.random.default_rng(side)
    dx = 1.0 / 128
    c = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 1, 3)
    x = ((40 + c + r.random((side ** 3, 8, 3)))).reshape(-1, 3)[:-3].astype(np.float32) * np.float32(dx)
    lam, mu = scenes.lame(1e4, 0.3)
    vol = dx ** 3 / 8
    m = scenes.ModelSpec(scenes.Material(scenes.FIXED_COROTATED, lam, mu), 1000 * vol, vol, x, np.zeros((1, 3), np.float32))
    return engine_from_scene(scenes.Scene("r", (32, 32, 32), (0, 0, 0), dx, -9.8, 1e-4, 0, [m]))


@pytest.mark.gpu
@pytest.mark.parametrize("side", [3, 22, 23])  # 213, 85k and 97k particles; 87,381 fit the staging
def test_positions_into_every_destination(side):
    import torch

    e = _engine(side)
    for k in range(2):
        e.Substep(0.0 if k == 0 else 1e-4, 1e-4)
    n = e.n(0)
    # the stored state, slot by slot: block-relative positions of the previous ordering
    st = e.state(0)[:3]
    keys, counts = e.layout(1)
    _, off = e.ordering(0, 1)
    want = np.empty((n, 3), np.float32)
    dx = np.float32(1.0 / 128)
    for j in range(counts[0]):
        b = np.array([keys[j] // 1024, keys[j] // 32 % 32, keys[j] % 32])
        s = slice(off[j], off[j + 1])
        want[s] = (4 * b).astype(np.float32) * dx + st[:, s].T
    lib = native.load()
    for pinned in (False, True):
        for shift in (0, 1, 5):
            buf = torch.full((3 * n + 16,), -7.0, pin_memory=pinned)
            p = ctypes.cast(buf.data_ptr() + 4 * shift, ctypes.POINTER(ctypes.c_float))
            cnt = ctypes.c_uint64()
            assert lib.ckmpm_get_positions(e._h, 0, p, n, ctypes.byref(cnt)) == native.OK and cnt.value == n
            got = buf.numpy()
            np.testing.assert_array_equal(got[shift:shift + 3 * n].reshape(n, 3), want)
            assert (got[:shift] == -7).all() and (got[shift + 3 * n:] == -7).all()
    c = e.counters()
    assert c.active_blocks == e.layout(0)[1][0] and c.flags == 0 and c.substeps == 2 and c.max_speed > 0
    e.close()
