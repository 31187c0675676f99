"""Rules that choose a kernel by sizes, and what the sampler is handed: what can be checked without a GPU."""

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


def test_sampler_takes_token_ids_of_any_kind():
    """Lists of Python's and numpy's integers, 0-d tensors, arrays and tensors of one id each; what is no id is refused."""
    from qwen25vl_lite_amd.sampling.sampler import _int32_ids
    for flat in ([3, 4], [np.int64(3), np.uint8(4)], list(torch.tensor([3, 4])), list(torch.tensor([[3], [4]])),
                 list(np.array([[3], [4]], np.int64)), ["3", 4]):
        got = _int32_ids(flat)
        assert got.dtype == np.int32 and got.tolist() == [3, 4], flat
    assert _int32_ids([]).tolist() == [0]
    for flat, error in (([1 << 40], OverflowError), ([np.int64(1 << 40)], OverflowError), ([None], TypeError),
                        (list(torch.tensor([[3, 4], [5, 6]])), (RuntimeError, TypeError, ValueError))):
        with pytest.raises(error):
            _int32_ids(flat)
