"""Products of 17 to 64 rows whose waves share K by halves (csrc/gemm_rows.hip), gated and cut along K: each against 64 bits."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = [17, 32, 33, 48, 49, 64]


def _operands(m, n, k, pad=0):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k + pad, device="cuda", generator=g).bfloat16()[:, :k]
    w = (torch.randn(n, k + pad, device="cuda", generator=g) / math.sqrt(k)).bfloat16()[:, :k]
    return x, w, x.double() @ w.double().T, k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)     # k roundings of a sum's terms


# channels of a group of waves on 256 compute units: one, four and five (one group of 8 rows, two), 9, 16, 21 and 24 (the most); inner sizes of one step
# part empty, of a half that has none of it, and off the steps
@pytest.mark.parametrize("channels, k, pad", [(8, 8, 0), (1024, 24, 8), (4096, 40, 0), (4104, 72, 0), (9216, 1000, 0), (16384, 136, 8),
                                              (20992, 64, 0), (24576, 256, 0)])
def test_gated(channels, k, pad):
    from qwen25vl_lite_amd.ops import rows
    for m in ROWS:
        x, w, z, off = _operands(m, 2 * channels, k, pad)
        for grouped in (True, False):
            gate, up = (z.view(m, -1, 2, 8)[:, :, i].reshape(m, -1) for i in (0, 1)) if grouped else z.chunk(2, 1)
            gate_off, up_off = (off.view(m, -1, 2, 8)[:, :, i].reshape(m, -1) for i in (0, 1)) if grouped else off.chunk(2, 1)
            if grouped:
                got, act = rows.rows_swiglu(x, w), torch.nn.functional.silu(gate)
                factor = up
            else:
                got = rows.rows_gated(x, w, 1.0, 2.0, 0.5)
                act = gate.clamp(max=2.0) * torch.sigmoid(gate.clamp(max=2.0))
                factor = up.clamp(-2.0, 2.0) + 0.5
            ref = act * factor
            # |silu'| < 1.1; float32 arithmetic of the activation: a few roundings of it, and of its argument in the exponent
            bound = (1.2 * gate_off * factor.abs() + act.abs() * up_off + 2.0 ** -20 * (1.0 + gate.abs()) * act.abs() * factor.abs()
                     + 2.0 ** -8 * ref.abs() + 1e-12)
            assert bool(((got.double() - ref).abs() <= bound).all()), (m, grouped)


@pytest.mark.parametrize("n, k, pad", [(1, 8, 0), (37, 264, 8), (127, 2056, 0), (129, 520, 0), (3584, 1032, 0), (6, 64 * 300 + 8, 0)])
def test_cut_along_the_inner_size(n, k, pad):
    """Slabs of blocks that are full, of one output, and of one more than a block's; a last range that is shorter."""
    from qwen25vl_lite_amd.ops import skinny
    for m in [9, 16] + ROWS:
        x, w, want, slack = _operands(m, n, k, pad)
        slabs = skinny.split_product(w, x)
        assert slabs.dim() == 3 and bool(((slabs.double().sum(0) - want).abs() <= slack).all()), m
