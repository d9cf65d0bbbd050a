"""The particle backward of one block split over up to 16 workgroups of 128 particles: at the
edges of chunks and splits, particles at one place have the velocity gradients of a single
particle of their mass (bar as for positions outside the block, tests/test_adjoint_far_sums.py)."""
import numpy as np
import pytest

from ckmpm_amd import scenes
from tests.test_adjoint_far_sums import _velocity_gradient


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 127, 128, 129, 256, 257, 1920, 2047, 2048, 2049, 4097, 30001])
def test_a_block_of_any_size(n):
    at = [4 * 7 + 1.75 + 2.3, 4 * 7 + 1.75 + 0.4, 4 * 7 + 1.75 + 3.1]
    one = _velocity_gradient(scenes.FIXED_COROTATED, 1, at, (0, 0, 0))
    many = _velocity_gradient(scenes.FIXED_COROTATED, n, at, (0, 0, 0))
    scale = np.abs(one).max()
    assert scale > 0
    assert np.abs(many - one).max() <= 1e-5 * scale, np.abs(many - one).max() / scale
