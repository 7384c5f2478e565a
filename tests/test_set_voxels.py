"""Many voxel writes in one call against the same writes one by one: sectors that share a place in the
call's table (128 voxels apart), rows that leave a sector and come back, repeated voxels, zeros, and
positions outside the scene, below zero too."""
from __future__ import annotations

import numpy as np
import pytest

from voxelrt_amd import Scene


def writes(kind, rng, size, ysize):
    if kind == "ball":
        g = np.stack(np.meshgrid(*[np.arange(-9, 10)] * 3, indexing="ij"), -1).reshape(-1, 3)
        return g[(g * g).sum(1) <= 81] + [33, 30, 63]
    if kind == "shared places":
        xyz = rng.integers(0, 32, (4000, 3))
        return xyz + rng.integers(0, 2, (4000, 3)) * [128, 128, 128]
    if kind == "outside":
        return rng.integers(-40, size + 40, (4000, 3))
    return rng.integers(0, [size, ysize, size], (4000, 3)) // rng.integers(1, 9)


@pytest.mark.parametrize("kind", ["ball", "shared places", "outside", "any"])
@pytest.mark.parametrize("size,ysize", [(32, 32), (256, 32), (256, 256)])
@pytest.mark.parametrize("n", [0, 1, 4000])
def test_set_voxels_equals_single_writes(kind, size, ysize, n):
    rng = np.random.default_rng(size + ysize + n)
    start = np.where(rng.random((ysize, size, size)) < 0.01, 3, 0).astype(np.uint8)
    one, many = Scene.from_dense(start), Scene.from_dense(start)
    xyz = writes(kind, rng, size, ysize)[:n].astype(np.int32)
    values = np.where(rng.random(len(xyz)) < 0.3, 0, rng.integers(1, 256, len(xyz))).astype(np.uint8)
    for (x, y, z), v in zip(xyz.tolist(), values.tolist()):
        one.set_voxel(x, y, z, v)
    many.set_voxels(xyz, values)
    assert one.dirty_sectors == many.dirty_sectors
    a, b = one.stream(), many.stream()
    assert all(np.array_equal(a[k], b[k]) for k in a if k != "_owner")
