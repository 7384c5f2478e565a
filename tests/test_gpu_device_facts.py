"""Facts about this part that the traversal's loops rest on (tests/hip/device_checks.hip)."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def checks(cuda):
    from voxelrt_amd import build

    lib = C.CDLL(str(build.CHECKS if build.CHECKS.exists() else build.build_checks()))
    P, u32 = C.c_void_p, C.c_uint32
    lib.check_structured_loads.argtypes = [P, u32, u32, P, u32, P, P]
    lib.check_take_slots.argtypes = [P, u32]
    lib.check_reciprocals.argtypes = [C.c_int, C.c_int, P, P]
    return lib


def test_structured_loads_up_to_4_gib(checks):
    """A structured load's index times its stride is right up to 2^32 - 1, past 2^31 too, and past the
    records it reads 0.  (From 2^32 on it is cut to 32 bits: the loops stay below, see masks_in_reach.)
    The table lies 2 GiB into its allocation, so that an offset taken as signed would read another of its
    entries."""
    pad, records = 1 << 28, (1 << 29) - 8
    buf = torch.empty(pad + records, dtype=torch.int64, device="cuda")
    want = [0, 1, (1 << 28) - 1, 1 << 28, (1 << 28) + 1, 3 << 27, records - 2, records - 1]
    for i in set(want) | {i - (1 << 29) for i in want if i >= 1 << 28}:
        buf[pad + i] = 1000003 * i + 17
    stream = torch.cuda.current_stream().cuda_stream
    table = buf[pad:].data_ptr()
    index = torch.tensor(want + [records, records + 7], dtype=torch.int32, device="cuda")
    out = torch.full((len(index),), -1, dtype=torch.int64, device="cuda")
    assert checks.check_structured_loads(table, 8, records, index.data_ptr(), len(index), out.data_ptr(), stream) == 0
    assert out.tolist() == [1000003 * i + 17 for i in want] + [0, 0]
    even = sorted({i & ~1 for i in want})  # the same bytes as records of 16
    for i in even:
        buf[pad + i] = 1000003 * i + 19
        buf[pad + i + 1] = -7 * i
    index = torch.tensor([i // 2 for i in even] + [records // 2], dtype=torch.int32, device="cuda")
    out = torch.full((len(index), 2), -1, dtype=torch.int64, device="cuda")
    assert checks.check_structured_loads(table, 16, records // 2, index.data_ptr(), len(index), out.data_ptr(),
                                         stream) == 0
    assert out.tolist() == [[1000003 * i + 19, -7 * i] for i in even] + [[0, 0]]
    del buf
    torch.cuda.empty_cache()


def test_reciprocal_in_range(checks):
    """reciprocal_in_range is 1 / x, correctly rounded, for every x with 2^-100 <= |x| < 2^101."""
    differ = torch.zeros(1, dtype=torch.int32, device="cuda")
    assert checks.check_reciprocals(-100, 100, differ.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    assert int(differ) == 0


def test_worlds_past_the_reach_of_structured_loads(vrt, checks):
    """A world whose bricks lie on both sides of slot 2^26, 4 GiB into the masks: every cast equals the same
    world's with its bricks in the first slots."""
    scene = vrt.Scene.spheres(14, 7, 600, 10.0, 30.0, 5)
    low = vrt.World.from_scene(scene)
    st = scene.stream()
    slots = (1 << 26) + (1 << 17)
    high = vrt.World(14, 7, initial_slots=slots, max_slots=slots)
    assert checks.check_take_slots(high.handle, (1 << 26) - 30000) == 0
    high.sync(st["sector_idx"], st["alloc_mask"], st["bricks"])
    palette = np.random.default_rng(4).integers(1, 1 << 40, 256).astype(np.uint64)
    for w in (low, high):
        w.set_palette(palette)
    assert high.info().slot_high_water > (1 << 26) + 10000
    assert low.info().slot_high_water < 1 << 17

    # rays to places in and around the bricks from up to 300 voxels away
    rng = np.random.default_rng(6)
    n = 300000
    si = rng.choice(st["sector_idx"], n).astype(np.int64)
    at = np.stack([si & 511, si >> 18, (si >> 9) & 511]) * 32.0 + rng.uniform(0, 32, (3, n))
    o = at + rng.normal(size=(3, n)) * rng.uniform(20, 150, (1, n))
    o[1] = np.clip(o[1], 0.5, 127.5)
    d = at - o
    d /= np.linalg.norm(d, axis=0)
    o, d = o.astype(np.float32), d.astype(np.float32)

    def same(a, b, what):
        assert torch.equal(a.rec, b.rec) and torch.equal(a.t, b.t) and torch.equal(a.pos, b.pos), what

    for count in (n, 100000, 3001):
        rays = vrt.RayBatch.from_numpy(np.ascontiguousarray(o[:, :count]), np.ascontiguousarray(d[:, :count]))
        for schedule, cap in ((1, 0), (2, 0), (3, 5)):
            a = low.cast(rays, schedule=schedule, pass_cap=cap, with_pos=True)
            same(high.cast(rays, schedule=schedule, pass_cap=cap, with_pos=True), a, ("cast", count, schedule))
            assert ((a.rec[:, 3] & 0xFF) != 0).any()
        for method in ("full", "coarse"):
            for lut in (False, True):
                same(high.cast_shader(rays, method, lut, with_pos=True),
                     low.cast_shader(rays, method, lut, with_pos=True), (method, lut, count))
    centre = at[:, 0]
    cam = vrt.CameraSpec((centre[0] + 40.0, 120.0, centre[2] + 40.0), 30.0, -40.0, 320, 200)
    for schedule in (1, 2):
        a, b = (vrt.cast_frame(w, cam, schedule=schedule, with_pos=True) for w in (low, high))
        assert all(torch.equal(x.rec, y.rec) and torch.equal(x.t, y.t) for x, y in zip(a, b))
    for lut in (False, True):
        a, b = (vrt.render_frame(w, cam, 2, 3, lut) for w in (low, high))
        assert torch.equal(a.albedo_normal, b.albedo_normal) and torch.equal(a.depth, b.depth)
        assert torch.equal(a.irradiance.view(torch.int32), b.irradiance.view(torch.int32))
    for tuning in ((8, 8, 1, 0), (8, 8, 2, 0)):
        recs = []
        for w in (low, high):
            batch = vrt.Batch([cam])
            vrt.BatchPlan(w, batch, tuning=tuning).launch()
            recs.append((batch.hits.rec, batch.hits.t))
        assert torch.equal(recs[0][0], recs[1][0]) and torch.equal(recs[0][1], recs[1][1]), tuning
    for k in range(20):
        args = (o[:, k].astype(np.float64), d[:, k].astype(np.float64))
        assert low.ray_cast(*args) == high.ray_cast(*args)
    high.close()
