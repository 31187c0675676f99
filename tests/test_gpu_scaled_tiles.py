"""Some hundred rows between the product that ends a mixer and the gated one behind the norm: the rows times the gain and their sums of squares that
csrc/gemm_mid.hip leaves, and csrc/gemm_tile.hip's products of such rows, each against 64 bits."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


# outputs for part of a block of 64, for one, for one more (rows that four does not divide among them), for blocks that the last XCDs have none of
@pytest.mark.parametrize("m, n, k, stride", [(1, 1, 32, 1), (65, 66, 160, 66), (80, 64, 128, 68), (81, 130, 96, 131), (300, 2048, 2048, 2048),
                                             (420, 2052, 256, 2056)])
def test_rows_left_for_the_norm(m, n, k, stride):
    from qwen25vl_lite_amd.ops import mid
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, device="cuda", generator=g).bfloat16()
    w = (torch.randn(n, k, device="cuda", generator=g) / math.sqrt(k)).bfloat16()
    gain, before = torch.randn(n, device="cuda", generator=g), torch.randn(m, stride, device="cuda", generator=g)
    plain, left = before.clone(), before.clone()
    assert mid.mid_into(plain[:, :n], x, w) is None
    rows, squares, parts = mid.mid_into(left[:, :n], x, w, gain)
    assert torch.equal(plain, left)
    assert torch.equal(rows, (left[:, :n] * gain).bfloat16())
    # sums of at most n squares, none negative: as many roundings at most
    exact = (left[:, :n].double() ** 2).sum(1)
    assert bool(((squares[:, :parts].double().sum(1) - exact).abs() <= n * 2.0 ** -24 * exact).all())


# every shape of tile, with rows and outputs for part of a tile and one more; one place of squares, places that four does not divide, all of them
@pytest.mark.parametrize("shape", range(10))
@pytest.mark.parametrize("m, n, k, parts, act", [(70, 272, 96, 1, "silu"), (257, 528, 128, 33, "gelu_tanh"), (321, 784, 2048, 256, "silu")])
def test_gated_rows_that_are_still_to_be_normed(shape, m, n, k, parts, act):
    from qwen25vl_lite_amd.ops import tile
    g, eps = torch.Generator(device="cuda").manual_seed(m + n + k), 1e-6
    h, gain = 3.0 * torch.randn(m, k, device="cuda", generator=g), torch.randn(k, device="cuda", generator=g)
    w = (torch.randn(n, k, device="cuda", generator=g) / math.sqrt(k)).bfloat16()
    rows = (h * gain).bfloat16()
    squares = torch.full((m, tile.PARTS), math.nan, device="cuda")
    pieces = (h * h).tensor_split(min(parts, k), dim=1)
    squares[:, :parts] = 0.0
    squares[:, :len(pieces)] = torch.stack([p.sum(1) for p in pieces], 1)
    out = tile.tile_swiglu(rows, w, act, shape=shape, scaled=(squares, parts, eps)).double()
    scale = 1.0 / torch.sqrt((h.double() ** 2).sum(1, keepdim=True) / k + eps)
    both = (rows.double() @ w.double().T * scale).view(m, n // 16, 2, 8)
    size = (rows.double().abs() @ w.double().abs().T * scale).view(m, n // 16, 2, 8)
    gate, up = both[:, :, 0], both[:, :, 1]
    acted = torch.nn.functional.silu(gate) if act == "silu" else torch.nn.functional.gelu(gate, approximate="tanh")
    # k roundings of a sum's terms, k of a row's squares and a few behind them; neither activation is steeper than 1.13; then one to bfloat16 and
    # a few units of the activation's exponential
    slack = (2 * k + 8) * 2.0 ** -24 * size
    want = (acted * up).reshape(m, n // 2)
    bound = (1.13 * slack[:, :, 0] * (up.abs() + slack[:, :, 1]) + acted.abs() * slack[:, :, 1]).reshape(m, n // 2)
    assert bool(((out - want).abs() <= bound + 2.0 ** -8 * want.abs() + 2.0 ** -18 * up.abs().reshape(m, n // 2) + 1e-30).all())
