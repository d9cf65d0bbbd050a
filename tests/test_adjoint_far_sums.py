"""Sums of velocity adjoints from positions outside their block's own cells (an imported state):
100,000 particles at one place pull at the same few nodes, and their gradients must be those
of a single particle of their mass.  Added up in FP64 they agree to a few FP32 roundings (bar
1e-5); 100,000 equal FP32 additions to one number lose 1e-4 and more."""
import numpy as np
import pytest

from ckmpm_amd import scenes
from ckmpm_amd.engine import engine_from_scene


def _velocity_gradient(kind, n, at, shift):
    g, dt = 64, 1e-3
    dx = 1.0 / g
    lam, mu = scenes.lame(1e4, 0.3)
    vol = dx ** 3 / 8
    x = np.tile(np.asarray(at, np.float64) * dx, (n, 1)).astype(np.float32)
    v = np.tile(np.array([0.3, -0.2, 0.1], np.float32), (n, 1))
    m = scenes.ModelSpec(scenes.Material(kind, lam, mu), 1000 * vol / n, vol / n, x, v)
    m.lam_p, m.mu_p = np.full(n, lam, np.float32), np.full(n, mu, np.float32)
    e = engine_from_scene(scenes.Scene("one", (16, 16, 16), (0, 0, 0), dx, 0.0, dt, 1, [m]), adjoint_segment=1)
    st = e.state(0)
    st[:3] += (np.asarray(shift) * dx).astype(np.float32)[:, None]
    e.set_state(0, st)
    e.adjoint_record(True)
    e.Substep(dt, dt)
    e.adjoint_record(False)
    e.Synchronize()
    e.adjoint_reset()
    e.adjoint_seed(0, np.tile(np.array([0.7, 0.45, -0.3], np.float32), (n, 1)))
    e.adjoint_substep()
    out = e.adjoint_gradients(0)[2]
    e.close()
    return out


# block faces lie at 4 k + 1.75: over the upper face in x, the lower one in y, an edge, a corner
@pytest.mark.gpu
@pytest.mark.parametrize("kind", [scenes.FIXED_COROTATED, scenes.NEO_HOOKEAN])
@pytest.mark.parametrize("shift", [(0.6, 0, 0), (0, -0.6, 0), (0.6, 0, 0.6), (-0.6, -0.6, -0.6), (0.6, 0.6, 0.6)])
def test_many_far_particles_are_one_heavy_one(kind, shift):
    at = [4 * 7 + 1.75 + (3.9 if s > 0 else 0.1 if s < 0 else 2.3) for s in shift]
    one = _velocity_gradient(kind, 1, at, shift)
    many = _velocity_gradient(kind, 100000, at, shift)
    scale = np.abs(one).max()
    assert scale > 0
    assert np.abs(many - one).max() <= 1e-5 * scale, np.abs(many - one).max() / scale
