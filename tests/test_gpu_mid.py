"""Products of some hundred rows in small tiles over all of the inner size (csrc/gemm_mid.hip): each against 64 bits."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


# one row, one row tile of either width (64 and 80 on 256 compute units), one row more; outputs for part of a block, for a block, for blocks that the
# last XCDs have none of; inner sizes of one step part empty, off the steps, and of one step more than are on their way
@pytest.mark.parametrize("m, n, k, pad", [(1, 1, 32, 0), (64, 64, 128, 0), (65, 70, 160, 8), (80, 520, 1056, 0), (81, 2048, 640, 0), (400, 3264, 96, 0),
                                          (300, 2048, 2048, 0)])
def test_added_to_the_residual(m, n, k, pad):
    from qwen25vl_lite_amd.ops import mid
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k + pad, device="cuda", generator=g).bfloat16()[:, :k]
    w = (torch.randn(n, k + pad, device="cuda", generator=g) / math.sqrt(k)).bfloat16()[:, :k]
    want, slack = x.double() @ w.double().T, k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)      # k roundings of a sum's terms
    for stride in (n, n + 3, n + 4):
        rows = torch.randn(m, stride, device="cuda")
        before, beside = rows[:, :n].double(), rows[:, n:].clone()
        mid.mid_into(rows[:, :n], x, w)
        total = before + want
        assert bool(((rows[:, :n].double() - total).abs() <= slack + 2.0 ** -23 * total.abs()).all()) and torch.equal(rows[:, n:], beside), stride


@pytest.mark.parametrize("m, k, nq, nkv, ps, bias", [(1, 32, 1, 1, 16, True), (65, 160, 3, 1, 16, True), (321, 416, 5, 2, 48, False), (81, 64, 4, 0, 16, True),
                                                     (420, 2048, 16, 2, 16, True), (129, 3072, 28, 4, 32, False)])
def test_projection_with_rotation_and_cache(m, k, nq, nkv, ps, bias):
    from qwen25vl_lite_amd.ops import mid
    from test_gpu_dispatch import _stacked_projection
    _stacked_projection(m, k, nq, nkv, 128, ps, bias, lambda x, w, b, cs, slots, kc, vc: mid.mid_heads(x, w, b, cs, slots, kc, vc, nq, nkv, ps))


def test_values_that_are_not_finite_stay_by_themselves():
    """One infinite and one undefined value channel: every other channel has the bits it has beside two channels of zeros."""
    from qwen25vl_lite_amd.ops import mid
    m, k, nq, nkv, ps = 70, 256, 2, 2, 16
    x, w = torch.randn(m, k, device="cuda").bfloat16(), (torch.randn((nq + 2 * nkv) * 128, k, device="cuda") / 16).bfloat16()
    cs, slots = torch.rand(m, 64, 2, device="cuda"), torch.arange(m, device="cuda", dtype=torch.int32)
    results = []
    for fill in ((0.0, 0.0), (math.inf, math.nan)):
        w[(nq + nkv) * 128 + 3], w[(nq + nkv + 1) * 128 + 73] = fill
        kc = torch.zeros(m // ps + 1, nkv, ps, 128, dtype=torch.bfloat16, device="cuda")
        vc = torch.zeros(m // ps + 1, nkv, 128, ps, dtype=torch.bfloat16, device="cuda")
        q = mid.mid_heads(x, w, None, cs, slots, kc, vc, nq, nkv, ps)
        results.append((q, kc, vc.permute(0, 3, 1, 2).reshape(-1, nkv * 128)[:m]))
    rest = torch.ones(nkv * 128, dtype=torch.bool, device="cuda")
    rest[[3, 128 + 73]] = False
    (q0, k0, v0), (q1, k1, v1) = results
    assert torch.equal(q0, q1) and torch.equal(k0, k1) and torch.equal(v0[:, rest], v1[:, rest])
