"""Products on both sides of the row counts and inner sizes at which another kernel takes over: each entry against 64 bits."""

import math
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = [1, 8, 9, 16, 17, 32, 33, 48, 49, 64, 65, 100]
INNER = [2040, 2048, 2056, 4104]


def _operands(m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, device="cuda", generator=g).bfloat16()
    w = (torch.randn(n, k, device="cuda", generator=g) / math.sqrt(k)).bfloat16()
    want = x.double() @ w.double().T
    return x, w, want, k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)     # k roundings of a sum's terms


@pytest.mark.parametrize("k", INNER)
@pytest.mark.parametrize("n", [272, 16400])
def test_products(n, k):
    """Few outputs and many (64 for each compute unit), plain, with a bias, in float32, joined to a sum."""
    from qwen25vl_lite_amd.ops import linear as products
    bias = torch.randn(n, device="cuda")
    for m in ROWS:
        x, w, want, slack = _operands(m, n, k)
        assert bool(((products.linear(x, w, out_dtype=torch.float32).double() - want).abs() <= slack).all()), m
        assert bool(((products.linear(x, w).double() - want).abs() <= slack + 2.0 ** -8 * want.abs()).all()), m
        got = products.linear(x, w, bias, out_dtype=torch.float32).double()
        total = want + bias.double()
        assert bool(((got - total).abs() <= slack + 2.0 ** -23 * (want.abs() + total.abs())).all()), m
        for residual in (None, torch.randn(m, n, device="cuda")):
            before = 0.0 if residual is None else residual.double()
            left = products.linear_into(residual, x, w)
            got = (before if left is None or residual is None else residual.double()) + (
                0.0 if left is None else left.double().sum(0) if left.dim() == 3 else left.double())
            if left is None:
                got = residual.double()
            last = 2.0 ** -8 if left is not None and left.dtype == torch.bfloat16 else 2.0 ** -23
            assert bool(((got - (want + before)).abs() <= slack + last * (want.abs() + (want + before).abs())).all()), m


@pytest.mark.parametrize("k", INNER)
@pytest.mark.parametrize("n", [272, 16400])
def test_gate_and_up(n, k):
    """Grouped and plain rows of gate and up, plain rows of x and rows whose norm may be formed on the way."""
    from qwen25vl_lite_amd.ops import linear as products
    gain = torch.rand(k, device="cuda") + 0.5
    for m in ROWS:
        x, w, want, slack = _operands(m, n, k)
        for grouped in (True, False):
            both, off = ((t.view(m, n // 16, 2, 8).transpose(1, 2).reshape(m, 2, n // 2) if grouped else t.view(m, 2, n // 2))
                         for t in (want, slack))
            # a product may be rounded to bfloat16 before the activation (whose slope is below 1.13)
            off = off + 2.0 ** -8 * (both.abs() + off)
            g, u = both[:, 0], both[:, 1]
            ref = torch.nn.functional.silu(g) * u
            bound = 1.13 * off[:, 0] * (u.abs() + off[:, 1]) + torch.nn.functional.silu(g).abs() * off[:, 1]
            got = products.gate_up_swiglu(x, w, grouped).double()
            assert bool(((got - ref).abs() <= bound + 2.0 ** -8 * (ref.abs() + bound)).all()), (m, grouped)
        h = torch.randn(m, k, device="cuda")
        lazy = products.NormedRows(h, gain, 1e-6, torch.bfloat16)
        x = lazy.materialize()
        got, ref = (products.gate_up_swiglu(t, w, True).double() for t in (lazy, x))
        # a normed value may be the neighbouring bfloat16, and so may a result
        moved = 2.0 ** -8 * (x.double().abs() @ w.double().abs().T)
        both, moved = ((t.view(m, n // 16, 2, 8).transpose(1, 2).reshape(m, 2, n // 2)) for t in (x.double() @ w.double().T, moved))
        bound = 1.13 * moved[:, 0] * (both[:, 1].abs() + moved[:, 1]) + (both[:, 0].abs() + moved[:, 0]) * moved[:, 1]
        assert bool(((got - ref).abs() <= bound + 2.0 ** -7 * ref.abs() + 1e-6).all()), m


@pytest.mark.parametrize("k", INNER)
def test_projection_with_rotation_and_cache(k):
    """The stacked projection of an attention: in one kernel with the rotation, cut along its inner size with the rotation's
    kernel adding the slabs, uncut.  Queries, keys and values against 64 bits, a token without a slot among them."""
    from qwen25vl_lite_amd.ops import kernels
    from qwen25vl_lite_amd.ops.linear import NormedRows
    from qwen25vl_lite_amd.parts import PartSpec, build_part
    nq, nkv, hd, ps = 4, 2, 32, 16
    part = build_part("mixer", PartSpec("paged_attention", {
        "hidden_size": k, "num_heads": nq, "num_kv_heads": nkv, "head_dim": hd, "qkv_bias": True,
        "position": PartSpec("rope", {"theta": 1e4})}), torch.bfloat16, torch.device("cuda:0"))
    torch.manual_seed(k)
    specs = part.param_specs()
    weights = {name: torch.randn(s.shape, device="cuda") / (math.sqrt(k) if len(s.shape) == 2 else 1.0) for name, s in specs.items()}
    part.load({name: t.bfloat16() if t.dim() == 2 else t for name, t in weights.items()})
    inv_freq, freq_row = part.position.rotary_tables(hd)
    gain = torch.rand(k, device="cuda") + 0.5
    for m in ROWS:
        h = torch.randn(m, k, device="cuda")
        lazy = NormedRows(h, gain, 1e-6, torch.bfloat16)
        x = lazy.materialize()
        pages = m // ps + 2
        slots = torch.randperm(pages * ps, device="cuda")[:m].int()
        if m > 2:
            slots[1] = -1
        group = SimpleNamespace(slot_mapping=slots, page_size=ps)
        positions = torch.randint(0, 900, (1, m), dtype=torch.int32, device="cuda")
        want = x.double() @ part.w_in.double().T + part.b_in.double()
        off = (k + 1) * 2.0 ** -24 * (x.double().abs() @ part.w_in.double().abs().T + part.b_in.double().abs())
        neighbour = 2.0 ** -8 * (x.double().abs() @ part.w_in.double().abs().T)   # norms formed in another order
        cs = kernels.rope_table(positions, inv_freq, freq_row, m).double()
        for rows in (x, lazy):
            if rows is lazy and m > 32:
                continue
            kc = torch.zeros(pages, nkv, ps, hd, dtype=torch.bfloat16, device="cuda")
            vc = torch.zeros(pages, nkv, hd, ps, dtype=torch.bfloat16, device="cuda")
            slot = SimpleNamespace(k_cache=kc, v_cache=vc)
            step = SimpleNamespace(positions=positions, per_pass={})
            args = (rows, step, group, slot, True, inv_freq, freq_row)
            q = part._project_few_rows(*args)
            if q is None:
                q = part._project(*args)

            def turned(t, bound):
                c, s = cs[:, None, :, 0], cs[:, None, :, 1]
                a, b = t[..., :hd // 2], t[..., hd // 2:]
                if bound:
                    c, s = c.abs(), s.abs()
                    return torch.cat([a * c + b * s, b * c + a * s], -1)
                return torch.cat([a * c - b * s, b * c + a * s], -1)
            slack = off + (neighbour if rows is lazy else 0.0)
            heads, bound = (t.view(m, nq + 2 * nkv, hd) for t in (want, slack))
            ref = torch.cat([turned(heads[:, :nq + nkv], False), heads[:, nq + nkv:]], 1)
            bound = torch.cat([turned(bound[:, :nq + nkv] + 2.0 ** -22 * heads[:, :nq + nkv].abs(), True), bound[:, nq + nkv:]], 1)
            bound = bound + 2.0 ** -8 * (ref.abs() + bound)
            assert bool(((q.view(m, nq, hd).double() - ref[:, :nq]).abs() <= bound[:, :nq]).all()), (m, rows is lazy)
            live = slots >= 0
            page, at = slots[live].long() // ps, slots[live].long() % ps
            keys, values = kc[page, :, at].double(), vc[page, :, :, at].double()
            assert bool(((keys - ref[live][:, nq:nq + nkv]).abs() <= bound[live][:, nq:nq + nkv]).all()), (m, rows is lazy)
            assert bool(((values - ref[live][:, nq + nkv:]).abs() <= bound[live][:, nq + nkv:]).all()), (m, rows is lazy)
            untouched = torch.ones(pages, ps, dtype=torch.bool, device="cuda")
            untouched[page, at] = False
            assert bool((kc.transpose(1, 2)[untouched] == 0).all()) and bool((vc.permute(0, 3, 1, 2)[untouched] == 0).all())


def _stacked_projection(m, k, nq, nkv, hd, ps, bias, call):
    """``call(x, w, bias, cs, slots, k cache, v cache)`` returns the rotated queries: these, keys and values against 64 bits, tokens without a
    slot among them; nothing else of the pages is written."""
    from qwen25vl_lite_amd.ops import kernels
    n, half = (nq + 2 * nkv) * hd, hd // 2
    torch.manual_seed(m + k)
    x, w = torch.randn(m, k, device="cuda").bfloat16(), (torch.randn(n, k, device="cuda") / math.sqrt(k)).bfloat16()
    b = torch.randn(n, device="cuda") if bias else None
    pages = m // ps + 2
    slots = torch.randperm(pages * ps, device="cuda")[:m].int()
    if m > 2:
        slots[1] = slots[m - 1] = -1
    kc = torch.zeros(pages, max(nkv, 1), ps, hd, dtype=torch.bfloat16, device="cuda")
    vc = torch.zeros(pages, max(nkv, 1), hd, ps, dtype=torch.bfloat16, device="cuda")
    positions = torch.randint(0, 900, (1, m), dtype=torch.int32, device="cuda")
    inv_freq = 1e4 ** (-torch.arange(0, hd, 2, device="cuda").float() / hd)
    cs = kernels.rope_table(positions, inv_freq, torch.zeros(half, dtype=torch.int32, device="cuda"), m)
    q = call(x, w, b, cs, *((slots, kc, vc) if nkv else (None, None, None)))
    want, off = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    if bias:
        want, off = want + b.double(), off + b.double().abs()
    want, off = want.view(m, -1, hd), ((k + 1) * 2.0 ** -24 * off).view(m, -1, hd)
    c, s = cs.double()[:, None, :, 0], cs.double()[:, None, :, 1]

    def turned(t, c, s, sign):
        return torch.cat([t[..., :half] * c - sign * t[..., half:] * s, t[..., half:] * c + t[..., :half] * s], -1)
    ref, bound = turned(want, c, s, 1.0), turned(off, c.abs(), s.abs(), -1.0)
    # two products and a sum in float32 each rounded, then bfloat16
    bound = bound + 2.0 ** -22 * turned(want.abs(), c.abs(), s.abs(), -1.0) + 2.0 ** -8 * ref.abs() + 1e-30
    assert bool(((q.view(m, nq, hd).double() - ref[:, :nq]).abs() <= bound[:, :nq]).all()), m
    if nkv:
        live = slots >= 0
        page, at = (slots[live] // ps).long(), (slots[live] % ps).long()
        assert bool(((kc[page, :, at].double() - ref[live][:, nq:nq + nkv]).abs() <= bound[live][:, nq:nq + nkv]).all()), m
        wv, ov = want[live][:, nq + nkv:], off[live][:, nq + nkv:]
        assert bool(((vc[page, :, :, at].double() - wv).abs() <= ov + 2.0 ** -8 * wv.abs() + 1e-30).all()), m
        untouched = torch.ones(pages, ps, dtype=torch.bool, device="cuda")
        untouched[page, at] = False
        assert bool((kc.transpose(1, 2)[untouched] == 0).all()) and bool((vc.permute(0, 3, 1, 2)[untouched] == 0).all())


@pytest.mark.parametrize("shape", [-1, 0, 1, 2, 3, 5, 8, 9])
@pytest.mark.parametrize("m, k, nq, nkv, ps, bias", [(65, 96, 3, 1, 16, True), (321, 160, 5, 2, 48, True), (129, 64, 4, 0, 16, False),
                                                     (256, 32, 1, 1, 32, False)])
def test_projection_of_many_rows_with_rotation_and_cache(m, k, nq, nkv, ps, bias, shape):
    """Every tile that holds both halves of a head, at rows, heads and inner sizes that leave the last tile and the last step part empty."""
    from qwen25vl_lite_amd.ops import tile
    _stacked_projection(m, k, nq, nkv, 128, ps, bias,
                        lambda x, w, b, cs, slots, kc, vc: tile.tile_heads(x, w, b, cs, slots, kc, vc, nq, nkv, ps, shape=shape))


@pytest.mark.parametrize("k, nq, nkv, hd, ps, bias", [(8, 3, 1, 10, 16, True), (2056, 5, 2, 48, 48, False), (3584, 28, 4, 128, 16, True),
                                                      (4096, 50, 7, 128, 32, True), (72, 64, 0, 128, 16, False), (3320, 1, 1, 2, 16, True)])
def test_projection_of_few_rows_in_slices(k, nq, nkv, hd, ps, bias):
    """Inner sizes that leave waves without any of it, one pair of channels a block and sixteen, rows on both sides of the column tiles."""
    from qwen25vl_lite_amd.ops import skinny
    for m in (1, 7, 8, 9, 16, 17, 32, 33, 48, 49, 64):
        _stacked_projection(m, k, nq, nkv, hd, ps, bias,
                            lambda x, w, b, cs, slots, kc, vc: skinny.slice_qkv_rope(w, cs, x, b, slots, kc, vc, nq, nkv, hd, ps))
    w = torch.empty(128, 4104, dtype=torch.bfloat16, device="cuda")
    assert not skinny.takes_slice(8, 4104, w, 32, 16, None) and not skinny.takes_slice(65, 4096, w[:, :4096], 32, 16, None)
    assert not skinny.takes_slice(8, 4096, w[:, :4096], 32, 8, None) and skinny.takes_slice(8, 4096, w[:, :4096], 32, 16, None)


@pytest.mark.parametrize("way", ["slices", "resident", "tiles"])
def test_values_that_are_not_finite_stay_by_themselves(way):
    """One infinite and one undefined value channel: every other channel of every head has the bits it has beside two channels of zeros."""
    from qwen25vl_lite_amd.ops import skinny, tile
    k, nq, nkv, hd, ps = 256, 2, 2, 128, 16
    n = (nq + 2 * nkv) * hd
    for m in (1, 17, 64) if way != "tiles" else (65,):
        torch.manual_seed(m)
        x, w = torch.randn(m, k, device="cuda").bfloat16(), (torch.randn(n, k, device="cuda") / 16).bfloat16()
        cs = torch.rand(m, hd // 2, 2, device="cuda")
        slots = torch.arange(m, device="cuda", dtype=torch.int32)
        bad = [(nq + nkv) * hd + 3, (nq + nkv + 1) * hd + hd // 2 + 9]
        results = []
        for fill in ((0.0, 0.0), (math.inf, math.nan)):
            w[bad[0]], w[bad[1]] = fill
            kc = torch.zeros(m // ps + 1, nkv, ps, hd, dtype=torch.bfloat16, device="cuda")
            vc = torch.zeros(m // ps + 1, nkv, hd, ps, dtype=torch.bfloat16, device="cuda")
            if way == "slices":
                q = skinny.slice_qkv_rope(w, cs, x, None, slots, kc, vc, nq, nkv, hd, ps)
            elif way == "tiles":
                q = tile.tile_heads(x, w, None, cs, slots, kc, vc, nq, nkv, ps)
            else:
                q = skinny.qkv_rope_product(w, cs, x=x, slots=slots, k_cache=kc, v_cache=vc, num_q_heads=nq, num_kv_heads=nkv,
                                            head_dim=hd, page_size=ps)
            v = vc.permute(0, 3, 1, 2).reshape(-1, nkv * hd)[:m]
            results.append((q, kc, v))
        (q0, k0, v0), (q1, k1, v1) = results
        rest = torch.ones(nkv * hd, dtype=torch.bool, device="cuda")
        rest[[3, hd + hd // 2 + 9]] = False
        assert torch.equal(q0, q1) and torch.equal(k0, k1) and torch.equal(v0[:, rest], v1[:, rest]), m
        assert not torch.isfinite(v1[:, ~rest]).any()


def test_which_projections_take_the_rotation_with_them():
    from qwen25vl_lite_amd.ops import kernels, tile
    w = torch.empty(4608, 3584, dtype=torch.bfloat16, device="cuda")
    x = torch.empty(2048, 3584, dtype=torch.bfloat16, device="cuda")
    assert tile.slab_ranges(x, w) == 1 and tile.prefers_heads(x, w, 1, 128, 64)
    assert tile.slab_ranges(x[:64], w) == 0 and not tile.prefers_heads(x[:64], w, 0, 128, 64)
    assert not tile.prefers_heads(x, w, 1, 128, 32) and not tile.prefers_heads(x, w, 1, 64, 32) and not tile.prefers_heads(x, w, 2, 128, 64)
    assert not tile.prefers_heads(x, w, 1, 128, 64, torch.empty(4609, device="cuda")[1:])
    if kernels.compute_units("cuda:0") == 256:
        assert tile.slab_ranges(x[:256], w) == 3


def test_projection_in_slabs_up_to_64_rows(monkeypatch):
    """As a large weight's, whose 49 to 64 rows are cut, too."""
    from qwen25vl_lite_amd.parts import attention
    monkeypatch.setattr(attention, "LARGE_WEIGHT", 0)
    test_projection_with_rotation_and_cache(4104)


@pytest.mark.parametrize("n, k, most", [(2048, 11008, 16), (2048, 16384, 16), (2048, 16392, 8), (3584, 18944, 8)])
def test_few_rows_cut_along_k(n, k, most):
    """Up to 8 rows, or 16 with a small weight, few ranges whose rows stay in their blocks; beyond, the streaming kernel's: as many
    slabs as the kernel that then runs writes, each against 64 bits in their sum."""
    from qwen25vl_lite_amd.ops import kernels, skinny
    cus = kernels.compute_units("cuda:0")
    for m in (1, 8, 9, 16, 17):
        x, w, want, slack = _operands(m, n, k)
        slabs = skinny.split_product(w, x)
        stem, name = ("gemm_resident", "qvl_gemm_split_chunks") if m <= most else ("gemm_rows", "qvl_gemm_rows_ranges")
        assert slabs.shape[0] == kernels._fn(stem, name, [skinny._c_int] * 4)(m, n, k, cus), m
        assert bool(((slabs.double().sum(0) - want).abs() <= slack).all()), m
