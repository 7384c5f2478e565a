"""Casts of few rays, a wave to each, around the count from which waves hold 64: records, positions and
counters equal to the persistent schedule's, and with a device count below the capacity."""
from __future__ import annotations

import pytest
import torch

from helpers import blob_world, random_rays

pytestmark = pytest.mark.gpu

PERSISTENT = 2


@pytest.fixture(scope="module")
def world(vrt):
    return vrt.World.from_scene(vrt.Scene.from_dense(blob_world(128, seed=9, density=0.01)))


@pytest.mark.parametrize("n", [1, 63, 64, 513, 4095, 4096, 4097])
@pytest.mark.parametrize("order", [0, 1])
def test_few_rays(vrt, cuda, world, n, order):
    rays = vrt.RayBatch.from_numpy(*random_rays(n, 128, seed=n, inside=False))
    count = torch.tensor([n - n // 3], dtype=torch.int32, device="cuda")
    for limit in (None, count):
        m = n if limit is None else int(limit)
        ca, cb = vrt.api.new_counters(), vrt.api.new_counters()
        a = world.cast(rays, with_pos=True, order=order, counters=ca, count=limit)
        b = world.cast(rays, with_pos=True, schedule=PERSISTENT, counters=cb, count=limit)
        assert torch.equal(a.rec[:m], b.rec[:m]) and torch.equal(a.t[:m], b.t[:m])
        assert torch.equal(a.pos[:, :m], b.pos[:, :m]) and torch.equal(ca, cb)


@pytest.mark.parametrize("n", [1, 4097, (1 << 19) - 1, 1 << 19, (1 << 19) + 65])
def test_compact_schedule_around_its_second_pass(vrt, cuda, world, n):
    rays = vrt.RayBatch.from_numpy(*random_rays(n, 128, seed=n, inside=False))
    want = world.cast(rays, with_pos=True, schedule=PERSISTENT)
    for cap in (0, 3, 32):
        got = world.cast(rays, with_pos=True, schedule=3, pass_cap=cap)
        assert torch.equal(got.rec, want.rec) and torch.equal(got.t, want.t) and torch.equal(got.pos, want.pos), cap
