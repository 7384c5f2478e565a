"""A world whose step table outgrows an L2, filled and emptied across the shares of sectors with bricks at
which casts change to the group table and back: records equal to the persistent schedule's each time."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import random_rays

pytestmark = pytest.mark.gpu


def test_casts_as_sectors_fill_and_empty(vrt, cuda):
    side = 64  # sectors, of 2048 voxels
    world = vrt.World(11, 11)
    rng = np.random.default_rng(3)
    order = rng.permutation(side**3).astype(np.uint32)
    rays = vrt.RayBatch.from_numpy(*random_rays((1 << 19) + 3, side * 32, seed=4, inside=True))
    held = 0
    for share in (0.02, 0.19, 0.21, 0.49, 0.51, 0.9, 0.3, 0.1, 0.0):
        want = int(share * side**3)
        idx = order[min(held, want):max(held, want)]
        # one brick each, or none
        bit = (np.uint64(1) << (idx.astype(np.uint64) % np.uint64(64))) * np.uint64(want > held)
        bricks = rng.integers(0, 2, (len(idx) if want > held else 0, 512), dtype=np.uint8)
        world.sync(idx, bit, bricks)
        held = want
        ref = world.cast(rays, schedule=2)
        for schedule in (1, 3):
            got = world.cast(rays, schedule=schedule)
            assert torch.equal(got.rec, ref.rec) and torch.equal(got.t, ref.t), (share, schedule)
