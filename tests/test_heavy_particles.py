"""Scenes in metres and tonnes from rest: the P2G accumulator's scale is largest where nothing
moves yet, and must leave the factors of heavy particles and wide cells finite.  In lockstep
with the FP64 oracle, with the bars of the small box scenes in units of the cell size."""
import numpy as np
import pytest

from ckmpm_amd import scenes
from ckmpm_amd.engine import engine_from_scene
from oracle.pyoracle import Oracle
from tests.test_gpu_parity import _box_scene, _compare_layout, _compare_ordering, _grid_close, _import

KINDS = [scenes.FIXED_COROTATED, scenes.NEO_HOOKEAN, scenes.DRUCKER_PRAGER, scenes.FLUID, scenes.VON_MISES,
         scenes.CAM_CLAY]


def _scaled(kind, dx, speed=0.0):
    sc = _box_scene(kind, seed=41 + kind, dim=8, speed=speed)
    m = sc.models[0]
    k = dx / sc.dx
    m.x = (m.x.astype(np.float64) * k).astype(np.float32)
    m.mass, m.volume = m.mass * k ** 3, m.volume * k ** 3
    sc.dx, sc.dt = dx, 1e-3 * dx  # sound at 10 to 20 m/s: 0.02 cells a substep
    return sc


def _lockstep(sc, steps):
    """Positions within 1e-5 dx, the other state within 2e-5, after every substep from the
    same inputs; the first with dt = 0, as the frame loop starts."""
    eng = engine_from_scene(sc)
    orc = Oracle.from_scene(sc)
    orc.setup()
    for k in range(steps):
        dt = 0.0 if k == 0 else sc.dt
        _import(eng, orc, 1)
        orc.physics(dt, sc.dt)
        eng.Substep(dt, sc.dt)
        eng.Synchronize()
        _grid_close(eng.grid_m(), orc.grid_mnext())
        sg, so = eng.global_state(0), orc.state_next(0)
        np.testing.assert_allclose(sg[:3], so[:3], rtol=0, atol=1e-5 * sc.dx)
        np.testing.assert_allclose(sg[3:], so[3:], rtol=0, atol=2e-5)
        orc.rebin([eng.state(0)[:3].T.copy()])
        _compare_layout(eng, orc, 0)
        _compare_ordering(eng, orc, 1)
    assert eng.counters().flags == 0 and orc.flags == 0
    eng.close()


# masses of 8 kg, 8 t (m dx = 2^15), 64 t, 1000 t; at 512 m the stress factor leads
@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("dx", [0.4, 4.0, 8.0, 20.0, 512.0])
def test_from_rest(kind, dx):
    _lockstep(_scaled(kind, dx), 4)


@pytest.mark.gpu
@pytest.mark.parametrize("dx", [4.0, 20.0])
def test_moving(dx):
    _lockstep(_scaled(scenes.NEO_HOOKEAN, dx, speed=0.3), 4)
