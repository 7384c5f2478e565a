"""The shader method's fast loop where it can go wrong, bit for bit against the oracle: worlds at and
under the 128 voxels it needs and of unequal heights, rays at the edge of what it takes, and the
level above empty sectors after edits that empty and fill sectors."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import blob_world
from test_gpu_fast_loop import edge_rays
from test_gpu_shader import MODES, check_mode
from test_oracle import dense_world

pytestmark = pytest.mark.gpu


def sparse_world(size, ysize, seed):
    vox = blob_world(size, seed=seed, density=0.0005, blobs=3, ysize=ysize)
    vox[ysize // 2:, : size // 2] = 0
    vox[:, :, size // 2:][:, : size // 4] = 0
    return vox


@pytest.mark.parametrize("size,ysize", [(64, 128), (128, 64), (128, 128), (256, 128), (128, 256)])
@pytest.mark.parametrize("origin", [(0, 0, 0), (5, -3, 17), (1 << 20, 64, -(1 << 20))])
def test_shader_loop_edges(vrt, oracle_mod, cuda, size, ysize, origin):
    vox = sparse_world(size, ysize, size + 3 * ysize)
    world = vrt.World.from_scene(vrt.Scene.from_dense(vox))
    ow = dense_world(oracle_mod, vox)
    for k, (o, d) in enumerate(edge_rays(2053, size, ysize, seed=size + ysize)):
        rel = (o.astype(np.float64) - np.array(origin, dtype=np.float64)[:, None]).astype(np.float32)
        for method, lut in MODES:
            for cap in (0, 1, 33):
                check_mode(world, ow, rel, d, origin, method, lut, f"set {k} origin {origin} cap {cap}", cap)


def test_levels_after_edits(vrt, oracle_mod, cuda):
    import oracle

    size = 256
    scene = vrt.Scene.from_dense(sparse_world(size, size, 5))
    world = vrt.World.from_scene(scene)
    rng = np.random.default_rng(6)
    (o, d), _, _ = edge_rays(4099, size, size, seed=7)
    for step in range(4):
        # a box of up to 100 voxels a side emptied, then one voxel set in each of a few sectors
        lo = rng.integers(0, size - 100, 3)
        ext = rng.integers(33, 100, 3)
        g = np.stack(np.meshgrid(*[np.arange(a, a + b) for a, b in zip(lo, ext)], indexing="ij"), -1).reshape(-1, 3)
        scene.set_voxels(g, 0)
        scene.delete_empty_bricks()
        scene.set_voxels(rng.integers(0, size, (5, 3)), 9)
        world.sync_scene(scene)
        ow = oracle.OracleWorld.from_stream(scene.stream())
        for method, lut in MODES:
            check_mode(world, ow, o, d, (0, 0, 0), method, lut, f"edit {step}")
