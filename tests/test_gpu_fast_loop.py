"""The casts' fast loop where it can go wrong, bit for bit against the oracle: worlds of one sector to
several groups of sectors and unequal heights, rays at the edge of what it takes (components near
2^-26 and nudged from zero, origins on and beside voxel planes, outside and far outside the world),
and world origins of every alignment and at its limit of 2^20."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import assert_hits_equal, blob_world, random_rays
from test_gpu_cast import gpu_cast, pair_from_dense

pytestmark = pytest.mark.gpu

ORIGINS = [(0, 0, 0), (5, -3, 17), (-32, 64, 32), (1 << 20, -(1 << 20), 3), (1 << 21, 0, 0)]


def edge_rays(n, size, ysize, seed):
    """Sets of n rays in world space: quick ones, nearly axis-aligned ones and far origins."""
    rng = np.random.default_rng(seed)
    box = np.array([[size], [ysize], [size]], dtype=np.float64)
    o, d = random_rays(n, size, seed, ysize=ysize, inside=False)
    sets = [(o, d)]
    # one or two components of 2^-26 to 2^-12, or nudged from zero; origins on planes, beside them, anywhere
    o = rng.uniform(0, 1, (3, n)) * box
    near = np.round(o) + rng.choice([0.0, 0.0, 1e-6, -1e-6, 1e-4, -1e-4, 0.5], (3, n))
    o = np.where(rng.random((3, n)) < 0.6, near, o)
    d = rng.normal(size=(3, n))
    d /= np.linalg.norm(d, axis=0)
    tiny = rng.choice([-1.0, 1.0], (3, n)) * 2.0 ** rng.uniform(-26, -12, (3, n))
    tiny = np.where(rng.random((3, n)) < 0.4, 2.0**-24, tiny)
    d = np.where(np.argsort(rng.random((3, n)), axis=0) < rng.integers(1, 3, (1, n)), tiny, d)
    sets.append((o, d / np.linalg.norm(d, axis=0)))
    # lengths of 0.3 to 3, origins up to 2^24 away and just outside the faces
    d = rng.normal(size=(3, n))
    d *= rng.uniform(0.3, 3.0, (1, n)) / np.linalg.norm(d, axis=0)
    far = rng.normal(size=(3, n)) * 2.0 ** rng.uniform(3, 24, (1, n))
    face = np.where(rng.random((3, n)) < 0.3, rng.choice([-1e-3, 0.0, 1e-3], (3, n)) + box * rng.integers(0, 2, (3, n)),
                    rng.uniform(0, 1, (3, n)) * box)
    sets.append((np.where(rng.random((1, n)) < 0.5, far, face), d))
    return [(np.ascontiguousarray(a, dtype=np.float32), np.ascontiguousarray(b, dtype=np.float32)) for a, b in sets]


@pytest.mark.parametrize("size,ysize", [(32, 32), (64, 32), (32, 128), (128, 64), (256, 128)])
@pytest.mark.parametrize("origin", ORIGINS)
def test_fast_loop_edges(vrt, oracle_mod, cuda, size, ysize, origin):
    vox = blob_world(size, seed=size + ysize, density=0.002, blobs=3, ysize=ysize)
    vox[ysize // 2:, : size // 2] = 0  # empty sectors and groups beside full ones
    world, ow = pair_from_dense(vrt, oracle_mod, vox)
    for k, (o, d) in enumerate(edge_rays(4099, size, ysize, seed=7 * size + ysize)):
        # relative to the world origin, rounded to f32 like a caller's
        rel = (o.astype(np.float64) - np.array(origin, dtype=np.float64)[:, None]).astype(np.float32)
        for max_iters in (1, 128):
            ref = ow.cast(rel, d, origin, max_iters, with_pos=True)
            for sched, cap in ((1, 0), (3, 3)):
                t, rec, pos = gpu_cast(world, rel, d, origin, max_iters, sched, cap, with_pos=True)
                what = f"set {k} origin {origin} cap {max_iters} schedule {sched}"
                assert_hits_equal(t, rec, ref["t"], ref["rec"], what)
                assert np.array_equal(t.view(np.uint32), ref["t"].view(np.uint32)), what
                hit = (rec[:, 3] & 0xFF) != 0
                assert np.array_equal(pos[:, hit].view(np.uint32), ref["pos"][:, hit].view(np.uint32)), what


@pytest.mark.parametrize("width,height,tile", [(40, 24, (8, 8)), (48, 8, (16, 4)), (37, 13, (1, 1)), (35, 21, (7, 3)),
                                               (64, 5, (64, 1))])
def test_tile_orders(vrt, cuda, width, height, tile):
    """Pixels of every tile shape: the device's rays equal the host's, whose tile order divides."""
    cam = vrt.CameraSpec((20.3, 40.7, 9.1), 33.0, -20.0, width, height, tile=tile)
    rb = cam.rays_device()
    o, d = cam.rays_host()
    assert np.array_equal(rb.d.cpu().numpy().view(np.uint32), d.view(np.uint32))
    assert np.array_equal(rb.o.cpu().numpy().view(np.uint32), o.view(np.uint32))
