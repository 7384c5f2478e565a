"""The brick-bucketed backward of gradients whose zeros need more lanes than a launch has (2^32, at a float4
each 68.7 GB): the split on the CPU, and such a gradient on the GPU."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

THREADS = 256


@pytest.mark.parametrize("blocks", [0, 1, 2**24 - 1, 2**24, 2**24 + 1, 2**25 - 2, 2**25 - 1, 3 * 2**37 // 1024 + 5])
def test_launches_cover_every_block(vrt, blocks):
    from voxelrt_amd import build

    lib = C.CDLL(str(build.CHECKS if build.CHECKS.exists() else build.build_checks()))
    lib.check_launches.argtypes = [C.c_uint64, C.c_uint32, C.c_void_p, C.c_uint32]
    each = np.zeros(64, dtype=np.uint32)
    n = lib.check_launches(blocks, THREADS, each.ctypes.data, len(each))
    assert int(each[:n].astype(np.uint64).sum()) == blocks
    assert n < len(each) and all(0 < int(b) * THREADS < 2**32 for b in each[:n])


@pytest.mark.gpu
def test_gradient_past_one_launch(vrt, cuda):
    import torch

    nvox = (2**34 + 2**20) // 3 + 1  # 2^32 float4s and some more, and floats after the last of them
    if torch.cuda.mem_get_info()[0] < nvox * 12 + (4 << 30):
        pytest.skip("needs 73 GB of device memory")
    vox = np.zeros((32, 32, 32), dtype=np.uint8)
    vox[3, 4, 5] = 1
    world = vrt.World.from_scene(vrt.Scene.from_dense(vox))
    ids = np.array([0, 511, 512, 2**31 - 1, 2**31, 2**32 - 3, 0], dtype=np.uint32)
    saved = torch.from_numpy(ids.view(np.int32)).cuda()
    grad_image = torch.arange(1, 22, dtype=torch.float32, device="cuda").reshape(7, 3)
    weight = torch.tensor([1.0, 2.0, 0.5, 4.0, 1.0, 8.0, 0.25], device="cuda")
    grad = vrt.render_backward(world, grad_image, saved, weight, nvox, mode="bricks")
    flat = grad.reshape(-1)
    want = {}
    for k, i in enumerate(ids.tolist()):
        for c in range(3):
            want[3 * i + c] = want.get(3 * i + c, 0.0) + float(weight[k]) * (3 * k + c + 1)
    assert all(float(flat[i]) == x for i, x in want.items())  # exact in f32
    step = 1 << 30
    assert sum(int(torch.count_nonzero(flat[i:i + step])) for i in range(0, flat.numel(), step)) == len(want)
    del grad, flat
    torch.cuda.empty_cache()
