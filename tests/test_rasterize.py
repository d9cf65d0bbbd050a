"""The setup's grid mass and momentum (RasterizeKernel) against an FP64 restatement: bodies
that touch faces, edges and corners of the blocks' reach, one velocity or one per particle,
several models on one grid, a block with a single particle."""
import numpy as np
import pytest

from ckmpm_amd import scenes
from ckmpm_amd.engine import engine_from_scene

G = 64
DX = 1.0 / G


def _grid(models, keys, nb):
    """M (nb, 4, 128) in FP64 from FP32 positions and velocities."""
    at = {int(k): i for i, k in enumerate(keys[:nb])}
    M = np.zeros((nb, 4, 128))
    for x, v, mass in models:
        xs = (x * np.float32(G)).astype(np.float64)
        for g, shift in ((0, 0.25), (1, -0.25)):
            c = np.floor((x * np.float32(G) + np.float32(shift)).astype(np.float64)).astype(int)
            t = xs - c + shift
            w0 = 1 - t + np.sin(2 * np.pi * t) / (2 * np.pi)
            for o in range(8):
                ov = np.array([o >> 2, (o >> 1) & 1, o & 1])
                w = np.where(ov, 1 - w0, w0).prod(1) * mass
                n = c + ov
                b, l = n // 4, n % 4
                key = (b[:, 0] * 16 + b[:, 1]) * 16 + b[:, 2]
                bi = np.array([at[int(k)] for k in key])
                node = g * 64 + l[:, 0] * 16 + l[:, 1] * 4 + l[:, 2]
                for ch, q in enumerate((w, w * v[:, 0], w * v[:, 1], w * v[:, 2])):
                    np.add.at(M, (bi, ch, node), q)
    return M


@pytest.mark.gpu
@pytest.mark.parametrize("per_particle", [False, True])
@pytest.mark.parametrize("counts", [(1,), (257, 3), (4000, 1500, 1)])
def test_setup_grid_matches_fp64(per_particle, counts):
    r = np.random.default_rng(len(counts))
    lam, mu = scenes.lame(1e4, 0.3)
    vol = DX ** 3 / 8
    models, specs = [], []
    for i, n in enumerate(counts):
        x = (14.0 + 4 * i + (9.0 if n > 100 else 2.0) * r.random((n, 3)))
        x[::5] = np.round(x[::5] * 4) / 4 + 0.75  # on the binning faces 4 k + 1.75 and on nodes
        x = (x * DX).astype(np.float32)
        v = (0.5 * r.standard_normal((n if per_particle else 1, 3))).astype(np.float32)
        specs.append(scenes.ModelSpec(scenes.Material(scenes.FIXED_COROTATED, lam, mu), 1000 * vol, vol, x, v))
        models.append((x, np.broadcast_to(v.astype(np.float64), (n, 3)), float(np.float32(1000 * vol))))
    e = engine_from_scene(scenes.Scene("r", (16, 16, 16), (0, 0, 0), DX, -9.8, 1e-4, 0, specs))
    keys, (_, nb, _) = e.layout(0)
    got = e.grid_m().astype(np.float64)
    want = _grid(models, keys, nb)
    # FP32 weights: each product carries a few 1e-7, of the largest node's value here
    for ch in range(4):
        assert np.abs(got[:, ch] - want[:, ch]).max() <= 2e-6 * np.abs(want[:, ch]).max()
    assert e.counters().flags == 0
    e.close()
