"""The brick-bucketed backward (vrt_render_bwd_bricks) on synthetic saved hits, against sums in 64
bits: pixel counts around a wave and a block, voxel counts that end inside a slot and inside a float4,
slots with one, few, many and no pixels, misses and zero weights."""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def small_world(vrt):
    vox = np.zeros((32, 32, 32), dtype=np.uint8)
    vox[3, 4, 5] = 1  # one brick: gradients of any size over 512 voxels
    return vrt.World.from_scene(vrt.Scene.from_dense(vox))


@pytest.mark.parametrize("npix", [1, 63, 64, 257, 5000, 300000])
@pytest.mark.parametrize("nvox", [512, 513, 5 * 512 + 77, 3001 * 512 + 2])
@pytest.mark.parametrize("spread", ["one slot", "few voxels", "all"])
def test_bricks_backward_sums(vrt, cuda, small_world, npix, nvox, spread):
    g = torch.Generator(device="cuda").manual_seed(npix * 31 + nvox)
    hi = {"one slot": 512, "few voxels": nvox, "all": nvox}[spread]
    voxel = torch.randint(0, hi, (npix,), generator=g, device="cuda")
    if spread == "few voxels":  # 7 voxels, the last among them
        some = torch.cat([torch.randint(0, nvox, (6,), generator=g, device="cuda"),
                          torch.tensor([nvox - 1], device="cuda")])
        voxel = some[torch.randint(0, 7, (npix,), generator=g, device="cuda")]
    weight = torch.rand(npix, generator=g, device="cuda") * 5
    weight[torch.rand(npix, generator=g, device="cuda") < 0.2] = 0.0
    miss = torch.rand(npix, generator=g, device="cuda") < 0.3
    saved = torch.where(miss, -1, voxel).to(torch.int32)
    grad_image = torch.randn((npix, 3), generator=g, device="cuda")
    got = vrt.render_backward(small_world, grad_image, saved, weight, nvox, mode="bricks")
    take = (~miss) & (weight != 0)
    each = torch.where(take[:, None], grad_image.double() * weight.double()[:, None], 0.0)
    want = torch.zeros((nvox, 3), dtype=torch.float64, device="cuda").index_add_(0, voxel, each)
    size = torch.zeros((nvox, 3), dtype=torch.float64, device="cuda").index_add_(0, voxel, each.abs())
    # each product and the sum are rounded once to 24 bits, the sum in between to 53
    assert bool(((got.double() - want).abs() <= 2.0**-23 * 1.001 * size).all())
    assert bool((got[size == 0] == 0).all())
