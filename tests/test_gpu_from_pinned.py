"""A step's integers out of pinned host memory by a kernel (csrc/elementwise.hip, qvl_from_host)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# part of a block of 1,024 words, all but its last pair, one, one pair more, many
@pytest.mark.parametrize("n", [2, 512, 1022, 1024, 1026, 34002])
def test_arrives_whole_each_time(n):
    from qwen25vl_lite_amd.ops.kernels import int32_from_pinned
    host, beside = torch.empty(n, dtype=torch.int32, pin_memory=True), torch.full((n + 8,), -7, dtype=torch.int32, device="cuda")
    out, came = beside[4:n + 4], torch.cuda.Event()
    for turn in range(3):                      # the same memory again, with other values: nothing of the last time's is kept anywhere
        host.random_(-2 ** 31, 2 ** 31 - 1)
        int32_from_pinned(host, out)
        came.record()
        came.synchronize()
        assert torch.equal(out.cpu(), host)
    assert bool((beside[:4] == -7).all()) and bool((beside[n + 4:] == -7).all())


def test_other_memory_is_refused():
    from qwen25vl_lite_amd.ops.kernels import KernelError, int32_from_pinned
    out = torch.empty(4, dtype=torch.int32, device="cuda")
    for host in (torch.zeros(4, dtype=torch.int32), torch.zeros(3, dtype=torch.int32, pin_memory=True), torch.zeros(4, dtype=torch.int64, pin_memory=True)):
        with pytest.raises(KernelError):
            int32_from_pinned(host, out if host.numel() == 4 else out[:3])
