"""Rules that choose a kernel by sizes: what can be checked without a GPU."""

import numpy as np
import pytest
import torch


@pytest.mark.parametrize("cus", [32, 64, 256])
@pytest.mark.parametrize("rows", [1, 8, 9, 64])
def test_products_are_cut_where_the_kernel_takes_the_cut(cus, rows, monkeypatch):
    """What takes_split accepts, the kernel behind it divides into ranges, on a device of any number of compute units (a part of
    one, say): the inner size may be as long as its blocks can keep."""
    from qwen25vl_lite_amd.ops import skinny
    monkeypatch.setattr(skinny, "_compute_units", lambda device: cus)
    taken = 0
    for k in [8, 4096, 4104, 2048 * cus - 8, 2048 * cus, 2048 * cus + 8, 4096 * cus, 4096 * cus + 8, 8192 * cus]:
        if skinny.takes_split(rows, k, torch.empty((3, k), dtype=torch.bfloat16)):
            taken += 1
            assert skinny._ranges(rows, 3, k, cus) > 0, k
    assert taken >= 5
