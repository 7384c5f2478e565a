"""The shader method from origins 2^16 to 2^28 voxels away, along each axis, by rays that are nearly
parallel to it and reach the world: bit for bit against the oracle.  rayCast's distances and its bias of
5 ulps are relative to the unclipped origin, so its positions step past the world's faces by tens of
voxels from 2^26 on; a world with bricks beside one face only shows a step that lands in another row's
sectors as a hit outside the world."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import blob_world
from test_gpu_shader import MODES, check_mode
from test_oracle import dense_world

pytestmark = pytest.mark.gpu


def far_rays(n, size, axis, sign, log2, seed):
    """Rays along `axis`, origins 2^log2[0] to 2^log2[1] before it, through points in and beside the world."""
    rng = np.random.default_rng(seed)
    p = rng.uniform(-4, size + 4, (3, n))
    r = 2.0 ** rng.uniform(log2[0], log2[1], n)
    d = rng.choice([-1.0, 1.0], (3, n)) * 2.0 ** rng.uniform(-22, -17, (3, n))
    beside = rng.random((3, n)) < 0.7  # origins beside the axis: the smallest |o| / |d| there
    d = np.where(beside, (p - rng.uniform(0, 4, (3, n))) / r, d)
    d[axis] = sign
    o = p - d * r
    o[axis] = -sign * r
    d = d * rng.uniform(0.6, 1.9, n)
    return np.ascontiguousarray(o, dtype=np.float32), np.ascontiguousarray(d, dtype=np.float32)


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("log2", [(16, 24), (23.9, 24.1), (24, 26), (26, 27), (27, 27.9)])
def test_far_origins(vrt, oracle_mod, cuda, axis, sign, log2):
    size = 256
    vox = blob_world(size, seed=11, density=0.002, blobs=3)
    vox[:, :32] = 0     # z < 32 empty, and x >= 64: bricks at the start of each row of sectors
    vox[:, :, 64:] = 0
    world = vrt.World.from_scene(vrt.Scene.from_dense(vox))
    ow = dense_world(oracle_mod, vox)
    o, d = far_rays(16384, size, axis, sign, log2, seed=int(10 * log2[1]) + axis)
    # waves in which every ray is one that the fast loop's bound on |o| / |d| takes, then all of them
    x = ((np.abs(o.astype(np.float64)) + 1) / np.abs(d)).sum(0) * np.linalg.norm(d, axis=0)
    quick = np.nonzero(x < 0.99 * 30 * 2.0**23)[0]
    assert quick.size > 1000
    order = np.concatenate([quick[: quick.size // 64 * 64], np.arange(o.shape[1])])
    o, d = np.ascontiguousarray(o[:, order]), np.ascontiguousarray(d[:, order])
    reached = 0
    for method, lut in MODES:
        rec = check_mode(world, ow, o, d, (0, 0, 0), method, lut, f"axis {axis} sign {sign} 2^{log2}")
        reached += int(((rec[:, 3] >> 16) & 0xFFFF > 0).sum())
    assert reached > 1000
