"""A world made on a stream that has long work queued, then filled and cast on another: its tables are
whole when its creation returns."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import assert_hits_equal, blob_world, random_rays
from test_oracle import dense_world

pytestmark = pytest.mark.gpu


def test_world_used_on_another_stream(vrt, oracle_mod, cuda):
    vox = blob_world(64, seed=51, density=0.01)
    scene = vrt.Scene.from_dense(vox)
    st = scene.stream()
    o, d = random_rays(5000, 64, seed=52, inside=False)
    rays = vrt.RayBatch.from_numpy(o, d)
    ref = dense_world(oracle_mod, vox).cast(o, d, (0, 0, 0), 128)
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    big = torch.zeros(1 << 26, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(first):
        for _ in range(100):  # some milliseconds
            big.add_(1.0)
    world = vrt.World(6, 6, stream=first)
    assert first.query()
    world.sync(st["sector_idx"], st["alloc_mask"], st["bricks"], stream=second)
    hits = world.cast(rays, 128, stream=second)
    shaded = world.cast_shader(rays, "full", True, stream=second)
    torch.cuda.synchronize()
    assert_hits_equal(hits.t.cpu().numpy(), hits.rec.cpu().numpy(), ref["t"], ref["rec"], "second stream")
    ref = dense_world(oracle_mod, vox).cast_shader(o, d, (0, 0, 0), "full", True)
    assert_hits_equal(shaded.t.cpu().numpy(), shaded.rec.cpu().numpy(), ref["t"], ref["rec"], "second stream, shader")
    # an empty world's casts miss on any stream
    with torch.cuda.stream(first):
        for _ in range(100):
            big.add_(1.0)
    empty = vrt.World(6, 6, stream=first)
    hits = empty.cast(rays, 128, stream=second)
    torch.cuda.synchronize()
    assert not bool(((hits.rec[:, 3] & 0xFF) != 0).any())
