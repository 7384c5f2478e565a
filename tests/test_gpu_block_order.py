"""Launches whose blocks are dispatched in windows of 512 (64 neighbours to an XCD): every ray of the
first, whole and last partial windows gets the record it gets without the windows, bit for bit."""
from __future__ import annotations

import pytest
import torch

from helpers import blob_world, random_rays

pytestmark = pytest.mark.gpu

PERSISTENT = 2
WINDOW = 64 * 512


@pytest.mark.parametrize("n", [WINDOW - 65, WINDOW - 63, WINDOW, WINDOW + 1, 2 * WINDOW, 3 * WINDOW + 64 * 7 + 5])
def test_windows_keep_every_ray(vrt, cuda, n):
    world = vrt.World.from_scene(vrt.Scene.from_dense(blob_world(128, seed=5, density=0.01)))
    o, d = random_rays(n, 128, seed=n, inside=False)
    rays = vrt.RayBatch.from_numpy(o, d)
    want = world.cast(rays, schedule=PERSISTENT)
    runs = {f"order {k}": world.cast(rays, order=k) for k in (0, 1)}
    batch = vrt.Batch([], [(0, n, (0, 0, 0), None)], rays)
    plan = vrt.BatchPlan(world, batch)
    plan.launch()
    runs["batch"] = batch.hits
    torch.cuda.synchronize()
    for what, h in runs.items():
        assert torch.equal(h.rec, want.rec) and torch.equal(h.t, want.t), what
    # the shader method: slices shorter than a window keep their blocks' order
    got, step = world.cast_shader(rays, "coarse", True), WINDOW - 64
    for at in range(0, n, step):
        part = vrt.RayBatch(rays.o[:, at:at + step].contiguous(), rays.d[:, at:at + step].contiguous(), (0, 0, 0))
        ref = world.cast_shader(part, "coarse", True)
        assert torch.equal(got.rec[at:at + step], ref.rec) and torch.equal(got.t[at:at + step], ref.t), at
