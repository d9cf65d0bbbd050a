"""G2P2G's LDS windows against the FP64 oracle, where its branches differ: positions outside
the block's own cells (an imported state), blocks of several rounds of 768 particles, and
blocks in which some particles move to another block while others of the same launch hold
none that does."""
import numpy as np
import pytest

from ckmpm_amd import scenes
from ckmpm_amd.engine import engine_from_scene
from oracle.pyoracle import Oracle
from tests.test_gpu_parity import (GRID_TOL, _box_scene, _compare_layout, _compare_ordering, _grid_close, _import,
                                   _lockstep)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [scenes.FLUID, scenes.NEO_HOOKEAN])
@pytest.mark.parametrize("shift", [-0.9, 0.9])
def test_positions_outside_the_blocks_cells(kind, shift):
    """Every particle shifted by 0.9 cells along each axis in the stored state: about
    two thirds then lie outside the cells 2..5 of their block, within the window [1,6].
    One substep from that state equals the oracle's, and so does the rebin after it."""
    sc = _box_scene(kind, seed=71, speed=0.0)
    eng = engine_from_scene(sc)
    orc = Oracle.from_scene(sc)
    orc.setup()
    eng.Substep(0.0, sc.dt)
    st = eng.state(0)
    st[:3] += np.float32(shift * sc.dx)
    eng.set_state(0, st)
    _import(eng, orc, 1)
    orc.physics(sc.dt, sc.dt)
    eng.Substep(sc.dt, sc.dt)
    eng.Synchronize()
    _grid_close(eng.grid_m(), orc.grid_mnext(), GRID_TOL)
    sg, so = eng.global_state(0), orc.state_next(0)
    np.testing.assert_allclose(sg[:3], so[:3], rtol=0, atol=2e-7)
    np.testing.assert_allclose(sg[3:], so[3:], rtol=0, atol=2e-5)
    orc.rebin([eng.state(0)[:3].T.copy()])
    _compare_layout(eng, orc, 0)
    _compare_ordering(eng, orc, 1)
    assert eng.counters().flags == 0


@pytest.mark.parametrize("speed", [0.0, 0.5])
def test_blocks_of_several_rounds(speed):
    """27 particles per cell: 1728 per block, three rounds; at rest no particle of a block
    moves, at 0.5 m/s some do in some rounds."""
    sc = _box_scene(scenes.NEO_HOOKEAN, seed=72, ppc_side=3, speed=speed)
    _lockstep(sc, 4, lambda k: (0.0 if k == 0 else sc.dt, sc.dt), (2e-7, 2e-5))
