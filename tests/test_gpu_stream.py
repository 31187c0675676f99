"""Products of up to 16 rows that go through K a share a wave (csrc/gemm_stream.hip), and the rows they leave for the norm behind them: each
against 64 bits."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = [1, 4, 5, 8, 9, 16]


def _operands(m, n, k, pad=0):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k + pad, device="cuda", generator=g).bfloat16()[:, :k]
    w = (torch.randn(n, k + pad, device="cuda", generator=g) / math.sqrt(k)).bfloat16()[:, :k]
    want = x.double() @ w.double().T
    return x, w, want, k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)     # k roundings of a sum's terms


# outputs a compute unit of 256: less than one, one, 8 and 9 (one item of either kind), 16 and 17 (one tile, two), 64 (the most); inner sizes that
# leave waves without any of it, and last groups of 64, 128 and 256 columns part empty; rows a multiple of 8 KB apart
@pytest.mark.parametrize("n, k, pad", [(1, 8, 0), (250, 72, 8), (2040, 1032, 0), (2304, 2056, 0), (4096, 520, 16), (4100, 3584, 0),
                                       (8192, 4096, 0), (16384, 136, 0), (2048, 11008, 0)])
def test_added_to_the_residual(n, k, pad):
    from qwen25vl_lite_amd.ops import stream
    gain = torch.randn(n, device="cuda")
    for m in ROWS:
        x, w, want, slack = _operands(m, n, k, pad)
        before = torch.randn(m, n + 4, device="cuda")
        plain, left = before.clone()[:, :n], before.clone()[:, :n]
        assert stream.stream_into(plain, x, w) is None
        rows, squares, parts = stream.stream_into(left, x, w, gain)
        total = before[:, :n].double() + want
        assert bool(((left.double() - total).abs() <= slack + 2.0 ** -23 * total.abs()).all()), m
        assert torch.equal(plain, left), m
        assert torch.equal(rows, (left * gain).bfloat16()), m
        # sums of at most n squares, none negative: as many roundings at most
        exact = (left.double() ** 2).sum(1)
        assert bool(((squares[:, :parts].double().sum(1) - exact).abs() <= n * 2.0 ** -24 * exact).all()), m
        if pad == 0:
            assert torch.equal(before[:, n:], torch.as_strided(left, (m, 4), (n + 4, 1), n)), m      # nothing beside the rows is written
    assert not stream.takes_into(17, k, w) and not stream.takes_into(1, k + 8, w)


@pytest.mark.parametrize("n, k", [(16, 8), (48, 200), (4096, 72), (4112, 1000), (22016, 2048), (37888, 640), (65536, 64), (8192 * 4, 4096)])
def test_gated_rows_that_are_still_to_be_normed(n, k):
    """One tile of channels a block to sixteen, some of them part empty, behind a norm that is not formed and behind none."""
    from qwen25vl_lite_amd.ops import stream
    eps = 1e-6
    for m in ROWS:
        x, w, _, _ = _operands(m, n, k)
        h, gain = torch.randn(m, k, device="cuda") * 3.0, torch.randn(k, device="cuda")
        parts = min(k, 200)
        squares = torch.full((m, stream.PARTS), math.nan, device="cuda")
        squares[:, :parts] = torch.stack([p.sum(1) for p in (h * h).tensor_split(parts, dim=1)], 1)
        for act in ("silu", "gelu_tanh"):
            for scaled in (None, (squares, parts, eps)):
                src = x if scaled is None else (h * gain).bfloat16()
                z, off = src.double() @ w.double().T, k * 2.0 ** -24 * (src.double().abs() @ w.double().abs().T)
                if scaled is not None:
                    by = torch.rsqrt((h.double() ** 2).sum(1, keepdim=True) / k + eps)
                    z, off = z * by, off * by + (k + 8) * 2.0 ** -24 * (z * by).abs()      # the squares' roundings, the root and its quotient
                z, off = z.view(m, n // 16, 2, 8), off.view(m, n // 16, 2, 8)
                a = torch.nn.functional.silu(z[:, :, 0]) if act == "silu" else torch.nn.functional.gelu(z[:, :, 0], approximate="tanh")
                ref = (a * z[:, :, 1]).reshape(m, n // 2)
                # |act'| < 1.13; float32 arithmetic of the activation: a few roundings of it, and of its argument in the exponent
                bound = (1.2 * off[:, :, 0] * z[:, :, 1].abs() + a.abs() * off[:, :, 1]
                         + 2.0 ** -20 * (1.0 + z[:, :, 0].abs()) * a.abs() * z[:, :, 1].abs()).reshape(m, n // 2) + 2.0 ** -8 * ref.abs() + 1e-12
                got = stream.stream_gated(src, w, act, scaled)
                assert bool(((got.double() - ref).abs() <= bound).all()), (m, act, scaled is not None)
    assert not stream.takes_gated(17, k, w) and not stream.takes_gated(1, k, w[:-8])


@pytest.mark.parametrize("k, nq, nkv, hd", [(264, 3, 1, 16), (2048, 16, 2, 128), (3584, 28, 4, 128), (4096, 8, 8, 128)])
def test_projection_of_rows_that_are_still_to_be_normed(k, nq, nkv, hd):
    """q | k | v of such rows: what the projection of the normed rows gives, up to the rounding of the rows."""
    from qwen25vl_lite_amd.ops import skinny, stream
    ps, eps, n = 16, 1e-6, (nq + 2 * nkv) * hd
    for m in ROWS:
        _, w, _, _ = _operands(m, n, k)
        h, gain, bias = torch.randn(m, k, device="cuda") * 2.0, torch.rand(k, device="cuda") + 0.5, torch.randn(n, device="cuda")
        rows = (h * gain).bfloat16()
        squares = torch.full((m, stream.PARTS), math.nan, device="cuda")
        squares[:, :3] = torch.stack([p.sum(1) for p in (h * h).tensor_split(3, dim=1)], 1)
        angle = torch.rand(m, hd // 2, device="cuda") * 6.0
        cs = torch.stack([angle.cos(), angle.sin()], -1).contiguous()
        slots = torch.arange(m, device="cuda", dtype=torch.int32)
        kc = torch.zeros(2, nkv, ps, hd, dtype=torch.bfloat16, device="cuda")
        vc = torch.zeros(2, nkv, hd, ps, dtype=torch.bfloat16, device="cuda")
        q = skinny.slice_qkv_rope(w, cs, rows, bias, slots, kc, vc, nq, nkv, hd, ps, (squares, 3, eps))
        by = torch.rsqrt((h.double() ** 2).sum(1, keepdim=True) / k + eps)
        z = (rows.double() @ w.double().T) * by
        off = (k + 8) * 2.0 ** -24 * (by * (rows.double().abs() @ w.double().abs().T) + bias.double().abs())
        z = (z + bias.double()).view(m, nq + 2 * nkv, hd)
        off = off.view(m, nq + 2 * nkv, hd)
        c, s = cs[..., 0].double()[:, None], cs[..., 1].double()[:, None]
        a, b = z[..., :hd // 2], z[..., hd // 2:]
        turned = torch.cat([a * c - b * s, b * c + a * s], -1)
        bound = 2.0 * (off + off.roll(hd // 2, -1)) + 2.0 ** -8 * turned.abs() + 2.0 ** -22 * (z.abs() + z.abs().roll(hd // 2, -1))
        assert bool(((q.view(m, nq, hd).double() - turned[:, :nq]).abs() <= bound[:, :nq]).all()), m
        keys = kc.transpose(1, 2).reshape(-1, nkv, hd)[:m].double()
        assert bool(((keys - turned[:, nq:nq + nkv]).abs() <= bound[:, nq:nq + nkv]).all()), m
        values = vc.permute(0, 3, 1, 2).reshape(-1, nkv, hd)[:m].double()
        assert bool(((values - z[:, nq + nkv:]).abs() <= off[:, nq + nkv:] + 2.0 ** -8 * z[:, nq + nkv:].abs()).all()), m
