"""The particle backward for positions outside their block's own cells (an imported state).
Two engines hold one layer of particles a hair on either side of a block face, so the blocks
differ while the grids agree; both import positions 0.6 cells above the face, inside the upper
engine's blocks and outside the lower one's.  Positions and gradients after two recorded
substeps agree to the hair (4e-5 cells, taken times the few-fold slopes of the weights)."""
import numpy as np
import pytest

from ckmpm_amd import scenes
from ckmpm_amd.engine import engine_from_scene


def _run(kind, hair):
    g, steps, dt = 64, 2, 1e-4
    dx = 1.0 / g
    r = np.random.default_rng(3)
    face = 4 * 7 + 1.75
    x = np.stack([np.full(600, face + hair), 20 + 10 * r.random(600), 20 + 10 * r.random(600)], 1) * dx
    x[:, 1:] += 0.02 * dx * ((x[:, 1:] / dx - 1.75) % 4 < 0.01)
    lam, mu = scenes.lame(1e4, 0.3)
    vol = dx ** 3 / 8
    v = 0.3 * r.standard_normal((600, 3))
    m = scenes.ModelSpec(scenes.Material(kind, lam, mu), 1000 * vol, vol, x.astype(np.float32), v.astype(np.float32))
    m.lam_p = (lam * (1 + 0.2 * r.random(600))).astype(np.float32)
    m.mu_p = (mu * (1 + 0.2 * r.random(600))).astype(np.float32)
    e = engine_from_scene(scenes.Scene("far", (16, 16, 16), (0, 0, 0), dx, -9.8, dt, steps, [m]), adjoint_segment=steps)
    st = e.state(0)
    st[0] += np.float32((0.6 - hair) * dx)
    e.set_state(0, st)
    blocks = e.layout(0)[0][: e.layout(0)[1][0]]
    e.adjoint_record(True)
    for _ in range(steps):
        e.Substep(dt, dt)
    e.adjoint_record(False)
    e.Synchronize()
    pos = e.positions_input_order(0) / dx
    e.adjoint_reset()
    e.adjoint_seed(0, r.standard_normal((600, 3)).astype(np.float32))
    for _ in range(steps):
        e.adjoint_substep()
    out = (pos,) + tuple(e.adjoint_gradients(0))
    e.close()
    return out, blocks


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [scenes.FIXED_COROTATED, scenes.NEO_HOOKEAN])
def test_far_positions_have_the_gradients_of_their_own_blocks(kind):
    (lo, keys_lo), (hi, keys_hi) = _run(kind, -2e-5), _run(kind, 2e-5)
    assert not np.intersect1d(keys_lo, keys_hi).size  # the lower engine's particles are all outside
    for a, b, name in zip(lo, hi, ("positions", "lambda", "mu", "velocity")):
        scale = np.abs(b).max()
        assert scale > 0, name
        assert np.abs(a - b).max() <= 1e-3 * scale, (name, np.abs(a - b).max(), scale)
