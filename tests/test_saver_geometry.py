"""The saver's memo of its paged caches, on the CPU: caches that are replaced are looked at
again, also where a new tensor takes the id of a freed one."""

from __future__ import annotations

import pytest
import torch

from marathon_amd import BlockShiftStore
from marathon_amd.connector import ShiftSaver

SHAPES = [(2, 4, 16, 8, 64), (4, 2, 16, 8, 64), (4, 8, 16, 128)]  # split planes, fused rows


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("inference", [True, False])
def test_replaced_caches_are_looked_at_again(shape, inference):
    saver = ShiftSaver(BlockShiftStore(64, "cpu"), 16)
    with torch.inference_mode(inference):  # there a view does not keep its base tensor
        for _ in range(20):
            kv = torch.zeros(shape)
            paged = saver._geometry([kv])[3]
            assert paged.first.data_ptr() == kv.data_ptr()
            del kv, paged
