"""Casts over the group table in worlds one to four sectors high, whose group words hold bits outside the
world: rays from inside, above and below, most of which leave through the top and bottom faces.  Records
equal to the persistent schedule's, which steps without the tables."""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# at least 2^18 sectors each; the grid takes the group table from four sectors of height on
@pytest.mark.parametrize("log2_y", [5, 6, 7, 8])
@pytest.mark.parametrize("share", [0.03, 0.18])
def test_flat_worlds(vrt, cuda, log2_y, share):
    log2_xz = 14
    nxz, ny = 1 << (log2_xz - 5), 1 << (log2_y - 5)
    rng = np.random.default_rng(8 * log2_y + int(100 * share))
    world = vrt.World(log2_xz, log2_y)
    idx = rng.permutation(nxz * nxz * ny)[:int(share * nxz * nxz * ny)].astype(np.uint32)
    bit = np.uint64(1) << (idx.astype(np.uint64) % np.uint64(64))
    world.sync(idx, bit, (rng.random((len(idx), 512)) < 0.3).astype(np.uint8))
    n = (1 << 19) + 77
    size = np.array([[1 << log2_xz], [1 << log2_y], [1 << log2_xz]], dtype=np.float64)
    o = rng.uniform(0, 1, (3, n)) * size
    o[:, :2000] = rng.uniform(-0.2, 1.2, (3, 2000)) * size
    o[1, 2000:4000] = rng.choice([0.0, float(1 << log2_y), 32.0], 2000)  # on the faces and a sector's plane
    d = rng.normal(size=(3, n))
    d[1] *= rng.choice([0.02, 0.2, 1.0], n)
    d /= np.linalg.norm(d, axis=0)
    for W in ((0, 0, 0), (3001, -7, 64)):
        rel = o - np.array(W, dtype=np.float64)[:, None]
        rays = vrt.RayBatch.from_numpy(rel.astype(np.float32), d.astype(np.float32), W)
        ref = world.cast(rays, schedule=2, with_pos=True)
        assert ((ref.rec[:, 3] & 0xFF) != 0).any()
        for schedule, cap in ((1, 0), (3, 0), (3, 3)):
            got = world.cast(rays, schedule=schedule, pass_cap=cap, with_pos=True)
            assert torch.equal(got.rec, ref.rec) and torch.equal(got.t, ref.t), (W, schedule, cap)
            assert torch.equal(got.pos, ref.pos), (W, schedule, cap)


@pytest.mark.parametrize("log2_xz,log2_y", [(13, 5), (12, 7), (5, 14), (8, 8)])
def test_tables_hold_the_world_and_its_border(vrt, cuda, log2_xz, log2_y):
    """Device memory of a world without bricks: the sector records, and two tables of 16-byte records with one
    sector of border around at least 4x4x4 sectors.  The rest (group words, palette, ray-cell table) is small."""
    nxz, ny = 1 << (log2_xz - 5), 1 << (log2_y - 5)
    tables = 16 * nxz * nxz * ny + 2 * 16 * (max(nxz, 4) + 2) ** 2 * (max(ny, 4) + 2)
    groups = 8 * (max(nxz // 4, 1) + 2) ** 2 * (max(ny // 4, 1) + 2) * 2
    info = vrt.World(log2_xz, log2_y).info()
    assert tables <= info.device_bytes <= tables + groups + 8192
