"""The pointers a ray batch passes on are those of its three component rows, whatever the tensors' strides."""
from __future__ import annotations

import pytest
import torch

from voxelrt_amd import RayBatch


@pytest.mark.parametrize("n", [0, 1, 5])
@pytest.mark.parametrize("form", ["whole", "rows of more", "columns of more", "expanded", "doubles"])
def test_ray_pointers(n, form):
    base = torch.zeros((7, n + 4), dtype=torch.float64 if form == "doubles" else torch.float32)
    t = {"whole": base[:3, :n].contiguous(), "rows of more": base[::2, :n], "columns of more": base[1:4, 3:3 + n],
         "expanded": base[0, :n].expand(3, n), "doubles": base[2:5, :n]}[form]
    rays = RayBatch(t, t.clone(), (1, -2, 3))
    want = [x[k].data_ptr() for x in (rays.o, rays.d) for k in range(3)]
    c, b = rays.to_c(), rays.buffers()
    for s in (c, b):
        assert [getattr(s, f) or 0 for f in ("ox", "oy", "oz", "dx", "dy", "dz")] == want
    assert list(c.world_origin) == [1, -2, 3] and c.n == n


def test_two_rows_are_refused():
    with pytest.raises(IndexError):
        RayBatch(torch.zeros((2, 4)), torch.zeros((3, 4)), (0, 0, 0)).to_c()
