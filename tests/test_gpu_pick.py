"""The picking cast (vrt_cast_one_f64) against the oracle where its kernel's prefetch and brick
masks can go wrong: worlds of one to many sectors, rays that cut sector corners, start outside,
run along an axis, have lengths other than 1, or run to the cap; and from several threads at once."""
from __future__ import annotations

import threading

import numpy as np
import pytest

from helpers import blob_world
from test_gpu_cast import pair_from_dense

pytestmark = pytest.mark.gpu


def pick_rays(n, size, ysize, seed):
    rng = np.random.default_rng(seed)
    o = rng.uniform(-0.2, 1.2, (n, 3)) * np.array([size, ysize, size])
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    d[: n // 4] = 0.0
    d[np.arange(n // 4), rng.integers(0, 3, n // 4)] = rng.choice([-1.0, 1.0], n // 4)  # along an axis
    o[n // 8: n // 4] = np.round(o[n // 8: n // 4])                                      # on voxel planes
    d[n // 4: n // 2] += rng.normal(scale=1e-9, size=(n // 2 - n // 4, 3))
    d[n // 2: n // 2 + n // 8] *= rng.uniform(0.01, 300.0, (n // 8, 1))
    return o, d


@pytest.mark.parametrize("size,ysize,max_iters", [(32, 32, 1024), (64, 128, 3), (128, 64, 1024), (256, 256, 400)])
def test_picks_match_oracle(vrt, oracle_mod, cuda, size, ysize, max_iters):
    world, ow = pair_from_dense(vrt, oracle_mod, blob_world(size, seed=size, density=0.001, blobs=3, ysize=ysize))
    for oo, dd in zip(*pick_rays(160, size, ysize, seed=size + 1)):
        g = world.ray_cast(oo, dd, max_iters)
        r = ow.cast_f64(oo, dd, max_iters)
        assert g.distance == r["distance"], (oo, dd)
        assert g.normal == tuple(r["normal"]) and g.uv == tuple(r["uv"]) and g.voxel_pos == tuple(r["voxel"]), (oo, dd)


def test_picks_from_threads(vrt, oracle_mod, cuda):
    worlds = [pair_from_dense(vrt, oracle_mod, blob_world(64, seed=s, density=0.01))[0] for s in (1, 2)]
    o, d = pick_rays(64, 64, 64, seed=3)
    want = [[w.ray_cast(a, b, 200) for a, b in zip(o, d)] for w in worlds]
    bad = []

    def picks(k):
        for i in range(64):
            j = (i * 7 + k) % 64
            w = (i + k) % 2
            if worlds[w].ray_cast(o[j], d[j], 200) != want[w][j]:
                bad.append((k, j))

    threads = [threading.Thread(target=picks, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
