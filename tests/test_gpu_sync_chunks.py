"""World syncs whose bricks, records and groups end around a staged chunk's edges and around the size
up to which kernels read the staging memory itself: the device's bricks and records afterwards."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_world import _device_bytes, sector_records

pytestmark = pytest.mark.gpu

CHUNK = ((8 << 20) - 256) // 516  # bricks of a full staging half
DIRECT = (4 << 20) // 516


@pytest.mark.parametrize("n", [1, 65, DIRECT - 40, DIRECT, CHUNK - 12, CHUNK - 1, CHUNK, CHUNK + 1, 2 * CHUNK + 3])
def test_sync_chunks(vrt, cuda, n):
    rng = np.random.default_rng(n)
    world = vrt.World(9, 9)
    for again in range(2):  # the second sync finds the staging halves in use
        nsec = -(-n // 64)
        idx = rng.permutation(4096)[:nsec].astype(np.uint32)
        mask = np.full(nsec, 2**64 - 1, dtype=np.uint64)
        mask[-1] = (1 << (n - 64 * (nsec - 1))) - 1 if n % 64 else 2**64 - 1
        bricks = rng.integers(0, 3, (n, 512), dtype=np.uint8)
        world.sync(idx, mask, bricks)
        rec, buf, info = sector_records(world), world.buffers(), world.info()
        vox = _device_bytes(buf.voxels, info.slot_capacity * 512).reshape(-1, 512)
        occ = _device_bytes(buf.occupancy, info.slot_capacity * 64).view(np.uint64).reshape(-1, 8)
        base = rec[idx.astype(np.int64), 2].astype(np.int64)
        assert np.array_equal(rec[idx.astype(np.int64), 0].astype(np.uint64)
                              | rec[idx.astype(np.int64), 1].astype(np.uint64) << np.uint64(32), mask)
        slots = np.concatenate([np.arange(64) + b for b in base])[:n]
        assert np.array_equal(vox[slots], bricks)
        # cell masks: bit vx + 4 vz + 16 vy of cell cx + 2 cz + 4 cy
        solid = (bricks != 0).reshape(n, 2, 4, 2, 4, 2, 4)  # cy vy cz vz cx vx
        bits = solid.transpose(0, 1, 3, 5, 2, 4, 6).reshape(n, 8, 64)
        want = (bits.astype(np.uint64) << np.arange(64, dtype=np.uint64)).sum(-1, dtype=np.uint64)
        assert np.array_equal(occ[slots], want)
