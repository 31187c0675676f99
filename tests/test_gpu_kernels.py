"""Each HIP kernel alone against a plain float32 formula, at sizes other than the engine's."""

import math

import pytest
import torch

from plain_model import (plain_apply_mrope, plain_attention, plain_inv_freq, plain_mrope_cos_sin, plain_rmsnorm)

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16]


def _tol(dtype):
    return dict(atol=1e-5, rtol=1e-5) if dtype == torch.float32 else dict(atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("dtype", DTYPES)
def test_embed_gather(dtype):
    from qwen25vl_lite_amd.ops import kernels
    torch.manual_seed(0)
    table = torch.randn(301, 100).to(dtype).cuda()
    ids = torch.tensor([0, 300, 7, 7, 150], dtype=torch.int32).cuda()
    out = kernels.embed_gather(ids, table)
    assert out.dtype == torch.float32 and torch.equal(out, table[ids.long()].float())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width, n", [(3584, 1), (8, 300), (2052, 19), (100, 3), (8192, 2)])
def test_embed_gather_with_rotation_tables(width, n, dtype):
    """Rows by 16 bytes and one by one, ids beyond the table's ends, scaled; beside them up to four rotation tables, the bits of a launch of
    their own."""
    from qwen25vl_lite_amd.ops import kernels
    torch.manual_seed(width)
    table = torch.randn(40, width).to(dtype).cuda()
    ids = torch.randint(-1, 41, (n,), dtype=torch.int32).cuda()
    positions = torch.randint(0, 5000, (3, n + 5), dtype=torch.int32).cuda()
    rotations = [(torch.rand(half).cuda(), torch.randint(-1, 3, (half,), dtype=torch.int32).cuda(), amplitude)
                 for half, amplitude in ((64, 1.0), (1, 0.5), (300, 1.25), (16, 1.0))]
    want = table[ids.long().clamp(0, 39)].float() * 1.5
    assert torch.equal(kernels.embed_gather(ids, table, scale=1.5), want)
    for count in (1, 3, 4):
        rows, tables = kernels.embed_gather(ids, table, scale=1.5, positions=positions, rotations=rotations[:count])
        assert torch.equal(rows, want) and len(tables) == count
        for got, (inv_freq, freq_row, amplitude) in zip(tables, rotations):
            assert torch.equal(got, kernels.rope_table(positions, inv_freq, freq_row, n, amplitude=amplitude))
    with pytest.raises(kernels.KernelError):
        kernels.embed_gather(ids, table, positions=positions, rotations=rotations + rotations[:1])


@pytest.mark.parametrize("width, slabs", [(4, 2), (1028, 1), (2048, 5), (3584, 17), (4096, 2), (4100, 9), (8192, 4)])
def test_add_rmsnorm_of_few_and_many_rows(width, slabs):
    """Both sides of the line between the kernels: the same bits for the same rows, and what float64 gives within the rounding of
    the slabs' sum (slabs + 1 additions) and of width squares, half an eps each at most, of which the root takes half."""
    from qwen25vl_lite_amd.ops import kernels
    torch.manual_seed(width)
    rows, eps = 513, 1e-6
    h, w = torch.randn(rows, width), torch.randn(width)
    delta = torch.randn(slabs, rows, width) if slabs > 1 else torch.randn(rows, width)
    total = h.double() + (delta.double().sum(0) if slabs > 1 else delta.double())
    want = total / torch.sqrt(total.pow(2).mean(1, keepdim=True) + eps) * w.double()
    hd = h.cuda()
    out = kernels.add_rmsnorm(hd, delta.cuda(), w.cuda(), eps, torch.float32)
    few_h, few_d = h[:40].contiguous().cuda(), (delta[:, :40] if slabs > 1 else delta[:40]).contiguous().cuda()
    few = kernels.add_rmsnorm(few_h, few_d, w.cuda(), eps, torch.float32)
    assert torch.equal(few, out[:40]) and torch.equal(few_h, hd[:40])
    eps32, size = 2.0 ** -23, (h.abs().double() + (delta.abs().double().sum(0) if slabs > 1 else delta.abs().double()))
    bound = (slabs + 1) * eps32 * size
    assert ((hd.cpu().double() - total).abs() <= bound).all()
    rel = bound.max() / total.pow(2).mean(1).sqrt().min() + (0.25 * width + 4) * eps32
    assert ((out.cpu().double() - want).abs() <= (bound + rel * total.abs()) / torch.sqrt(total.pow(2).mean(1, keepdim=True)) * w.abs().double()).all()


@pytest.mark.parametrize("width, slabs", [(256, 17), (1024, 16), (5120, 3), (5124, 1), (6144, 2), (6148, 1), (7168, 5), (7172, 1)])
def test_add_rmsnorm_of_few_and_many_rows_of_other_widths(width, slabs):
    """Rows that leave waves of the slabs' kernel without a piece, and all numbers of pieces of many wide rows."""
    test_add_rmsnorm_of_few_and_many_rows(width, slabs)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width", [16, 2052, 3584])
def test_embed_gather_on_both_sides_of_many_rows(width, dtype):
    from qwen25vl_lite_amd.ops import kernels
    torch.manual_seed(width)
    table = torch.randn(30, width).to(dtype).cuda()
    for n in (255, 256):
        ids = torch.randint(0, 30, (n,), dtype=torch.int32).cuda()
        assert torch.equal(kernels.embed_gather(ids, table, scale=0.5), table[ids.long()].float() * 0.5)


@pytest.mark.parametrize("width", [97, 3584, 8200])
@pytest.mark.parametrize("delta_dtype, out_dtype", [(torch.float32, torch.float32), (torch.float32, torch.bfloat16),
                                                    (torch.bfloat16, torch.bfloat16), (None, torch.bfloat16)])
def test_add_rmsnorm(width, delta_dtype, out_dtype):
    from qwen25vl_lite_amd.ops import kernels
    torch.manual_seed(width)
    n, eps = 5, 1e-5
    h = torch.randn(n, width) * 3
    delta = torch.randn(n, width).to(delta_dtype) if delta_dtype is not None else None
    w = 1 + 0.1 * torch.randn(width)
    total = h + (delta.float() if delta is not None else 0)
    want = plain_rmsnorm(total, w, eps)
    hd = h.cuda()
    out = kernels.add_rmsnorm(hd, None if delta is None else delta.cuda(), w.cuda(), eps, out_dtype)
    assert out.dtype == out_dtype
    assert torch.allclose(out.float().cpu(), want, **_tol(out_dtype))
    assert torch.allclose(hd.cpu(), total, atol=1e-6), "the sum is written back in float32"
    # selected rows: h stays as it was
    hd = h.cuda()
    rows = torch.tensor([4, 0, 4], dtype=torch.int32).cuda()
    out = kernels.add_rmsnorm(hd, None if delta is None else delta.cuda(), w.cuda(), eps, out_dtype, rows=rows)
    assert torch.allclose(out.float().cpu(), want[[4, 0, 4]], **_tol(out_dtype)) and torch.equal(hd.cpu(), h)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq, nkv, hd, sections, ps", [(6, 2, 24, (4, 4, 4), 16), (5, 1, 48, (10, 6, 8), 16),
                                                       (4, 4, 128, (16, 24, 24), 16), (6, 2, 24, (4, 4, 4), 48),
                                                       (4, 4, 128, (16, 24, 24), 32)])
def test_rope_kv_write(dtype, nq, nkv, hd, sections, ps):
    from qwen25vl_lite_amd.ops import kernels
    torch.manual_seed(hd)
    n, pages, theta = 11, 5, 1e4
    x = torch.randn(n, (nq + 2 * nkv) * hd)
    bias = torch.randn((nq + 2 * nkv) * hd) * 0.1
    pos = torch.stack([torch.randint(0, 5000, (n,)) for _ in range(3)])
    slots = torch.randperm(pages * ps)[:n].to(torch.int32)
    inv = plain_inv_freq(hd, theta)
    rows = torch.tensor(sum(([r] * c for r, c in enumerate(sections)), []), dtype=torch.int32)
    kc = torch.zeros(pages, nkv, ps, hd, dtype=dtype).cuda()
    vc = torch.zeros(pages, nkv, hd, ps, dtype=dtype).cuda()
    q = kernels.rope_kv_write(x.cuda(), bias.cuda(), pos.to(torch.int32).cuda(), inv.cuda(), rows.cuda(), slots.cuda(),
                              kc, vc, nq, nkv, hd, ps, out_dtype=dtype)
    xb = x + bias
    qs, ks, vs = xb.split([nq * hd, nkv * hd, nkv * hd], dim=1)
    cos, sin = plain_mrope_cos_sin(pos, inv)
    qr, kr = plain_apply_mrope(qs.view(n, nq, hd).transpose(0, 1), ks.view(n, nkv, hd).transpose(0, 1), cos, sin, sections)
    tol = dict(atol=2e-4, rtol=1e-4) if dtype == torch.float32 else _tol(dtype)   # sin/cos of angles up to 5000
    assert torch.allclose(q.float().cpu().view(n, nq, hd), qr.transpose(0, 1), **tol)
    kflat = kc.float().cpu().permute(0, 2, 1, 3).reshape(pages * ps, nkv, hd)          # [slot, kv head, hd]
    vflat = vc.float().cpu().permute(0, 3, 1, 2).reshape(pages * ps, nkv, hd)
    assert torch.allclose(kflat[slots.long()], kr.transpose(0, 1), **tol)
    assert torch.allclose(vflat[slots.long()], vs.view(n, nkv, hd), **_tol(dtype))
    untouched = torch.ones(pages * ps, dtype=torch.bool)
    untouched[slots.long()] = False
    assert kflat[untouched].abs().max() == 0 and vflat[untouched].abs().max() == 0
    # with the step's table of cosines and sines in hand the kernel gives the very same values
    cs = kernels.rope_table(pos.to(torch.int32).cuda(), inv.cuda(), rows.cuda(), n)
    want_cs = torch.stack([torch.cos(pos[rows.long()].T.float() * inv), torch.sin(pos[rows.long()].T.float() * inv)], dim=-1)
    assert torch.allclose(cs.cpu(), want_cs, atol=2e-4)
    kc2, vc2 = torch.zeros_like(kc), torch.zeros_like(vc)
    q2 = kernels.rope_kv_write(x.cuda(), bias.cuda(), pos.to(torch.int32).cuda(), inv.cuda(), rows.cuda(), slots.cuda(),
                               kc2, vc2, nq, nkv, hd, ps, out_dtype=dtype, cs=cs)
    if dtype == torch.float32:
        assert torch.equal(q2, q) and torch.equal(kc2, kc) and torch.equal(vc2, vc)
    else:   # float32 sums to bfloat16 with the table: the kernel with 16-byte loads
        for a, b in ((q2, q), (kc2, kc), (vc2, vc)):
            assert torch.allclose(a.float(), b.float(), atol=2e-2, rtol=1e-2)
        assert torch.equal(vc2, vc)
    # position 0 leaves a head as it is; a negative slot writes nothing; rot < hd leaves the tail alone
    kc.zero_()
    q0 = kernels.rope_kv_write(x.cuda(), None, torch.zeros(3, n, dtype=torch.int32).cuda(), inv.cuda(), rows.cuda(),
                               torch.full((n,), -1, dtype=torch.int32).cuda(), kc, vc, nq, nkv, hd, ps, out_dtype=dtype)
    assert torch.allclose(q0.float().cpu(), x[:, :nq * hd].to(dtype).float(), atol=1e-6) and kc.abs().max() == 0
    half = hd // 4
    qp = kernels.rope_kv_write(x[:, :nq * hd].contiguous().cuda(), None, pos.to(torch.int32).cuda(),
                               plain_inv_freq(2 * half, theta).cuda(), torch.zeros(half, dtype=torch.int32).cuda(),
                               None, None, None, nq, 0, hd, ps, out_dtype=dtype)
    qp = qp.float().cpu().view(n, nq, hd)
    assert torch.allclose(qp[..., 2 * half:], x[:, :nq * hd].view(n, nq, hd)[..., 2 * half:].to(dtype).float(), atol=1e-6)
    c1, s1 = plain_mrope_cos_sin(pos[:1].expand(3, n), plain_inv_freq(2 * half, theta))
    want, _ = plain_apply_mrope(x[:, :nq * hd].view(n, nq, hd)[..., :2 * half].transpose(0, 1),
                                x[:, :nq * hd].view(n, nq, hd)[..., :2 * half].transpose(0, 1), c1, s1, (half, 0, 0))
    assert torch.allclose(qp[..., :2 * half], want.transpose(0, 1), **tol)


def test_rope_kv_write_from_slabs():
    """The projection as slabs of partial sums: the rotation's kernel adds them in order and gives
    what it gives for their sum."""
    from qwen25vl_lite_amd.ops import kernels
    torch.manual_seed(3)
    n, nq, nkv, hd, ps, pages = 40, 6, 2, 48, 16, 9
    cols = (nq + 2 * nkv) * hd
    slabs = torch.randn(3, n, cols).cuda()
    total = slabs[0] + slabs[1]
    total = total + slabs[2]
    bias = torch.randn(cols).cuda()
    pos = torch.randint(0, 500, (3, n), dtype=torch.int32).cuda()
    inv_freq = plain_inv_freq(hd, 10000.0).cuda()
    freq_row = torch.tensor([0] * 8 + [1] * 8 + [2] * 8, dtype=torch.int32).cuda()
    slots = torch.randperm(pages * ps)[:n].to(torch.int32).cuda()
    cs = kernels.rope_table(pos, inv_freq, freq_row, n)
    outs = []
    for x in (slabs, total):
        kc = torch.zeros(pages, nkv, ps, hd, dtype=torch.bfloat16).cuda()
        vc = torch.zeros(pages, nkv, hd, ps, dtype=torch.bfloat16).cuda()
        q = kernels.rope_kv_write(x, bias, pos, inv_freq, freq_row, slots, kc, vc, nq, nkv, hd, ps,
                                  out_dtype=torch.bfloat16, cs=cs)
        outs.append((q, kc, vc))
    for a, b in zip(*outs):
        assert torch.equal(a, b)
    assert outs[0][0].abs().sum() > 0 and outs[0][1].abs().sum() > 0
    with pytest.raises(kernels.KernelError):      # slabs are taken with the table in hand only
        kernels.rope_kv_write(slabs, bias, pos, inv_freq, freq_row, slots, outs[0][1], outs[0][2], nq, nkv, hd, ps,
                              out_dtype=torch.bfloat16)


@pytest.mark.parametrize("n", [1, 40, 520])
@pytest.mark.parametrize("count", [2, 9, 10, 17])
def test_rope_kv_write_adds_any_number_of_slabs(count, n):
    """One batch of slabs that are asked for together, several, the last one partly filled; tokens that share the device's blocks
    and a block each; rotation of a part of the head, tokens without a slot: the bits of the slabs' sum taken in order."""
    from qwen25vl_lite_amd.ops import kernels
    torch.manual_seed(count + n)
    nq, nkv, hd, ps, half, pages = 6, 2, 48, 16, 16, n // 16 + 2
    cols = (nq + 2 * nkv) * hd
    slabs = torch.randn(count, n, cols).cuda()
    total = slabs[0]
    for s in slabs[1:]:
        total = total + s
    bias = torch.randn(cols).cuda()
    pos = torch.randint(0, 500, (1, n), dtype=torch.int32).cuda()
    inv_freq = plain_inv_freq(2 * half, 10000.0).cuda()
    freq_row = torch.zeros(half, dtype=torch.int32).cuda()
    slots = torch.randperm(pages * ps)[:n].to(torch.int32)
    slots[1::7] = -1
    slots = slots.cuda()
    cs = kernels.rope_table(pos, inv_freq, freq_row, n)
    outs = []
    for x in (slabs, total):
        kc = torch.full((pages, nkv, ps, hd), 7.0, dtype=torch.bfloat16).cuda()
        vc = torch.full((pages, nkv, hd, ps), 7.0, dtype=torch.bfloat16).cuda()
        q = kernels.rope_kv_write(x, bias, pos, inv_freq, freq_row, slots, kc, vc, nq, nkv, hd, ps,
                                  out_dtype=torch.bfloat16, cs=cs)
        outs.append((q, kc, vc))
    for a, b in zip(*outs):
        assert torch.equal(a, b)
    # what is not turned is the sum with the bias, rounded once
    plain = (total + bias).bfloat16().view(n, nq + 2 * nkv, hd)
    q, kc, vc = outs[0]
    assert torch.equal(q.view(n, nq, hd)[..., 2 * half:], plain[:, :nq, 2 * half:])
    live = slots >= 0
    page, at = slots[live].long() // ps, slots[live].long() % ps
    assert torch.equal(kc[page, :, at][..., 2 * half:], plain[live][:, nq:nq + nkv, 2 * half:])
    assert torch.equal(vc[page, :, :, at], plain[live][:, nq + nkv:])
    free = torch.ones(pages, ps, dtype=torch.bool, device="cuda")
    free[page, at] = False
    assert bool((kc.transpose(1, 2)[free] == 7.0).all()) and bool((vc.permute(0, 3, 1, 2)[free] == 7.0).all())


def _paged(k, v, ps, pages, dtype, seed):
    """Scatter per-request keys/values [nkv, T, hd] into shuffled pages; returns caches and tables."""
    g = torch.Generator().manual_seed(seed)
    nkv, hd = k[0].shape[0], k[0].shape[2]
    kc = torch.randn(pages, nkv, ps, hd, generator=g).to(dtype)          # stale values everywhere
    vc = torch.randn(pages, nkv, hd, ps, generator=g).to(dtype)
    order = torch.randperm(pages, generator=g).tolist()
    width = max((x.shape[1] + ps - 1) // ps for x in k)
    table = torch.full((len(k), width), -1, dtype=torch.int32)
    for r, (kr, vr) in enumerate(zip(k, v)):
        for i in range((kr.shape[1] + ps - 1) // ps):
            page = order.pop()
            table[r, i] = page
            n = min(ps, kr.shape[1] - i * ps)
            kc[page, :, :n] = kr[:, i * ps:i * ps + n].to(dtype)
            vc[page, :, :, :n] = vr[:, i * ps:i * ps + n].transpose(1, 2).to(dtype)
    return kc, vc, table


# the last shape has more query heads to a key/value head (20) than a column tile has columns: a
# token's heads span two tiles
ATTN_SHAPES = [(6, 2, 24, None), (5, 1, 48, 40), (8, 8, 16, 7), (14, 2, 128, None), (4, 2, 80, 130), (40, 2, 64, None)]


def _attention_case(dtype, nq, nkv, hd, window, lens=(333, 17, 64, 1), qlens=(5, 17, 1, 1), ps=16):
    """Prompt portions and single tokens of several requests in one call, pages shuffled, stale
    values in every unused slot.  One query and one far key are scaled so that a single score
    dominates: a kernel that misses that key (a page, a window edge) fails by far."""
    torch.manual_seed(nq * hd)
    lens, qlens = list(lens), list(qlens)   # context of each request after this step; its last qlen tokens are this step's
    last = lens[0] - 1
    k = [torch.randn(nkv, t, hd).to(dtype).float() for t in lens]
    v = [torch.randn(nkv, t, hd).to(dtype).float() for t in lens]
    q_all = [torch.randn(nq, t, hd) for t in lens]
    far = 2 if window is None else max(0, last - window + 1)      # the first key the last query still sees
    kf = k[0][:, far].repeat_interleave(nq // nkv, 0)
    q_all[0][:, last] = kf * (30.0 / (kf.pow(2).sum(-1, keepdim=True) * hd ** -0.5))      # that score is 30
    q_all = [x.to(dtype).float() for x in q_all]
    scale = hd ** -0.5
    kc, vc, table = _paged(k, v, ps, sum((t + ps - 1) // ps for t in lens) + 11, dtype, 1)
    qs, req, seqpos, want = [], [], [], []
    for r, (t, ql) in enumerate(zip(lens, qlens)):
        full = plain_attention(q_all[r], k[r], v[r], scale, window)      # [nq, t, hd]
        for p in range(t - ql, t):
            qs.append(q_all[r][:, p].reshape(-1))
            req.append(r)
            seqpos.append(p)
            want.append(full[:, p].reshape(-1))
    want = torch.stack(want)
    # the dominated row (request 0, its last position) really is the far key's value
    assert torch.allclose(want[qlens[0] - 1].view(nq, hd), v[0][:, far].repeat_interleave(nq // nkv, 0), atol=1e-3)
    return dict(q=torch.stack(qs).to(dtype).cuda(), kc=kc.cuda(), vc=vc.cuda(), table=table.cuda(),
                req=torch.tensor(req, dtype=torch.int32).cuda(), seqpos=torch.tensor(seqpos, dtype=torch.int32).cuda(),
                want=want, scale=scale, lens=lens, qlens=qlens)


# other page sizes than 16 (the reference tests 32, reference tests/test_paged_attn_kernel.py:89);
# 48 is the one where a 32-key block straddles pages at changing places
PAGE_SIZES = [(14, 2, 128, None, 32), (5, 1, 48, 40, 48), (4, 2, 80, 130, 64), (6, 2, 24, None, 32), (14, 2, 128, 70, 48),
              (7, 1, 128, None, 64)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq, nkv, hd, window, ps", [(*s, 16) for s in ATTN_SHAPES] + PAGE_SIZES)
def test_paged_attention_generic(dtype, nq, nkv, hd, window, ps):
    from qwen25vl_lite_amd.ops import kernels
    c = _attention_case(dtype, nq, nkv, hd, window, ps=ps)
    out = kernels.paged_attention_generic(c["q"], c["kc"], c["vc"], c["table"], c["req"], c["seqpos"], nq, window,
                                          c["scale"])
    tol = dict(atol=2e-5, rtol=1e-4) if dtype == torch.float32 else dict(atol=1.5e-2, rtol=2e-2)
    assert torch.allclose(out.float().cpu(), c["want"], **tol), (out.float().cpu() - c["want"]).abs().max()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq, nkv, hd, vd, ps, window, keep, chunk", [
    (4, 2, 128, 128, 16, None, 0, None), (4, 2, 100, 132, 4, None, 0, None), (3, 1, 36, 20, 12, 150, 5, None),
    (4, 4, 4, 512, 8, 64, 130, None), (2, 1, 64, 64, 16, None, 0, 130), (4, 2, 30, 24, 16, 150, 5, None), (4, 2, 32, 24, 6, None, 0, 90)])
def test_generic_attention_of_long_contexts(dtype, nq, nkv, hd, vd, ps, window, keep, chunk):
    """More blocks of 64 keys than waves, blocks skipped between kept keys and a window, the last block short; head and page sizes the
    wide loads take and do not take.  Every slot that a token does not see holds NaN."""
    from qwen25vl_lite_amd.ops import kernels
    torch.manual_seed(nq + hd + vd)
    n, length = 5, 601
    pages = (length + ps - 1) // ps
    seen = torch.zeros(n, length, dtype=torch.bool)
    at = [600, 300, 63, 64, 0]
    for i, p in enumerate(at):
        lo = max(0, p - window + 1) if window else 0
        lo = max(lo, p - p % chunk) if chunk else lo
        seen[i, lo:p + 1] = True
        seen[i, :min(keep, lo)] = True
    q, sinks = torch.randn(n, nq, hd).to(dtype), torch.randn(nq)
    k, v = torch.randn(n, nkv, length, hd).to(dtype), torch.randn(n, nkv, length, vd).to(dtype)
    kc = torch.full((n * pages, nkv, ps, hd), math.nan, dtype=dtype)
    vc = torch.full((n * pages, nkv, vd, ps), math.nan, dtype=dtype)
    table = torch.randperm(n * pages).view(n, pages).to(torch.int32)
    for i in range(n):
        for j in torch.nonzero(seen[i]).flatten().tolist():
            kc[table[i, j // ps], :, j % ps] = k[i, :, j]
            vc[table[i, j // ps], :, :, j % ps] = v[i, :, j]
    got = kernels.paged_attention_generic(q.reshape(n, -1).cuda(), kc.cuda(), vc.cuda(), table.cuda(), torch.arange(n, dtype=torch.int32).cuda(),
                                          torch.tensor(at, dtype=torch.int32).cuda(), nq, window, hd ** -0.5, keep_first=keep,
                                          chunk=chunk, sinks=sinks.cuda())
    per = nq // nkv
    s = torch.einsum("nhd,nhtd->nht", q.double(), k.double().repeat_interleave(per, 1)) * hd ** -0.5
    s = torch.cat([s.masked_fill(~seen[:, None], -math.inf), sinks.double().view(1, nq, 1).expand(n, nq, 1)], 2)
    want = torch.einsum("nht,nhtd->nhd", torch.softmax(s, 2)[:, :, :length], v.double().repeat_interleave(per, 1)).reshape(n, -1)
    tol = dict(atol=2e-5, rtol=1e-4) if dtype == torch.float32 else dict(atol=1.5e-2, rtol=2e-2)
    assert torch.allclose(got.double().cpu(), want, **tol), (got.double().cpu() - want).abs().max()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hd, vd", [(256, 256), (64, 129), (64, 257), (8, 511)])
def test_generic_attention_of_wide_values(dtype, hd, vd):
    """Values of more channels than are read at a time, the last ones alone."""
    test_generic_attention_of_long_contexts(dtype, 2, 1, hd, vd, 8, 150, 5, None)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hd, vd, window, keep, chunk", [(64, 64, 16, 0, None), (16, 24, 1, 0, None), (100, 132, 20, 12, None), (32, 260, 33, 0, None),
                                                         (64, 64, 40, 24, None), (128, 128, 64, 0, None), (64, 64, None, 0, 24), (64, 200, None, 0, 50),
                                                         (8, 8, 30, 0, 17)])
def test_generic_attention_of_few_keys(dtype, hd, vd, window, keep, chunk):
    """Windows and chunks of so few keys that one wave looks at them, or two, the kept ones among them."""
    test_generic_attention_of_long_contexts(dtype, 4, 2, hd, vd, 8, window, keep, chunk)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("hd", [64, 62])
@pytest.mark.parametrize("low", [(64, 128), (0, 64), (0, 256), (130, 301)])
def test_generic_attention_beside_scores_of_minus_infinity(dtype, hd, low):
    """Keys whose scores overflow to minus infinity, whole blocks of them, have no weight beside others: wherever the blocks stand
    among those that the waves share, with and without a sink."""
    from qwen25vl_lite_amd.ops import kernels
    g = torch.Generator().manual_seed(hd + low[0])
    length, ps = 301, 16
    q = torch.full((1, 1, hd), 1e20).to(dtype)
    k = torch.randn(length, hd, generator=g) * 1e-20
    k[low[0]:low[1]] = -1e20
    k, v = k.to(dtype), torch.randn(length, hd, generator=g).to(dtype)
    pages = (length + ps - 1) // ps
    kc, vc = torch.zeros(pages, 1, ps, hd, dtype=dtype), torch.zeros(pages, 1, hd, ps, dtype=dtype)
    for j in range(length):
        kc[j // ps, 0, j % ps], vc[j // ps, 0, :, j % ps] = k[j], v[j]
    s = (k.double() @ q[0, 0].double()) * hd ** -0.5
    for sinks in (None, torch.tensor([0.5])):
        terms = s if sinks is None else torch.cat([s, sinks.double()])
        want = torch.softmax(terms, 0)[:length] @ v.double()
        got = kernels.paged_attention_generic(q.reshape(1, -1).cuda(), kc.cuda(), vc.cuda(), torch.arange(pages, dtype=torch.int32).view(1, -1).cuda(),
                                              torch.zeros(1, dtype=torch.int32).cuda(), torch.tensor([length - 1], dtype=torch.int32).cuda(), 1,
                                              None, hd ** -0.5, sinks=None if sinks is None else sinks.cuda())
        tol = dict(atol=2e-5, rtol=1e-4) if dtype == torch.float32 else dict(atol=1.5e-2, rtol=2e-2)
        assert torch.allclose(got[0].double().cpu(), want, **tol), (sinks, (got[0].double().cpu() - want).abs().max())


@pytest.mark.parametrize("split", ["tile", "tile_two_groups", "coop", "coop_split", "coop_split_two_kernels"])
@pytest.mark.parametrize("nq, nkv, hd, window, ps", [(*s, 16) for s in ATTN_SHAPES if s[2] % 16 == 0]
                         + [s for s in PAGE_SIZES if s[2] % 16 == 0])
def test_paged_attention_matrix_cores(nq, nkv, hd, window, ps, split, monkeypatch):
    """The matrix-core kernels on the same case: blocks that own several tiles and share the keys
    through LDS (one group of waves, or two that take the key blocks in turn and merge), the waves
    of a block sharing one tile, and the keys further split among blocks, whose partial results the
    last block to finish merges (or a second kernel, for callers without counters)."""
    from qwen25vl_lite_amd.ops import attention_mfma
    from qwen25vl_lite_amd.parts import StepContext
    c = _attention_case(torch.bfloat16, nq, nkv, hd, window, ps=ps)
    plan = {"tile": ("tile", 1, 0), "tile_two_groups": ("tile", 1, 0), "coop": ("coop", 1, 0),
            "coop_split": ("coop", 6, 64), "coop_split_two_kernels": ("coop", 6, 64)}[split]
    if split == "coop_split_two_kernels":
        monkeypatch.setattr(attention_mfma, "MERGE_COUNTERS", 0)
    groups = {"tile": 1, "tile_two_groups": 2}.get(split)
    if groups == 2 and hd > 128:
        pytest.skip("two groups of waves are built for head sizes up to 128")
    monkeypatch.setattr(attention_mfma, "plan_splits", lambda t, n, m, d=None: plan)
    cu = [0]
    for ql in c["qlens"]:
        cu.append(cu[-1] + ql)
    none = torch.zeros(0, dtype=torch.int32).cuda()
    step = StepContext(num_tokens=cu[-1], num_reqs=4, token_ids=none, positions=none, token_req=c["req"],
                       token_seqpos=c["seqpos"], cu_q=torch.tensor(cu, dtype=torch.int32).cuda(),
                       ctx_len=torch.tensor(c["lens"], dtype=torch.int32).cuda(), req_slots=none, groups=[],
                       logit_rows=none, cu_q_host=cu, ctx_len_host=c["lens"], max_q_len=17, max_ctx_len=333,
                       dtype=torch.bfloat16)
    out = attention_mfma.try_attention(c["q"], c["kc"], c["vc"], c["table"], step, nq, window, c["scale"],
                                       force_groups=groups)
    assert out is not None
    err = (out.float().cpu() - c["want"]).abs().max()
    assert torch.allclose(out.float().cpu(), c["want"], atol=1.5e-2, rtol=2e-2), err
    if split == "coop_split":
        # the counters are back at zero, and a second launch right behind the first finds them so
        again = attention_mfma.try_attention(c["q"], c["kc"], c["vc"], c["table"], step, nq, window, c["scale"])
        assert torch.equal(again, out)
        torch.cuda.synchronize()
        assert int(attention_mfma._counters(c["q"].device).abs().sum()) == 0


@pytest.mark.parametrize("split", ["coop", "coop_split", "coop_split_two_kernels"])
@pytest.mark.parametrize("nq, nkv, hd, window", [(14, 2, 128, None), (6, 2, 48, 100), (8, 8, 16, 7)])
def test_a_step_of_decoded_tokens_only(nq, nkv, hd, window, split, monkeypatch):
    """Every request brings one token: the kernel is not handed the lists of tiles and of run
    starts (tile i is request i's, its token is token i) and gives what it gives with them."""
    from qwen25vl_lite_amd.ops import attention_mfma
    from qwen25vl_lite_amd.parts import StepContext
    lens = (333, 17, 64, 1, 200)
    c = _attention_case(torch.bfloat16, nq, nkv, hd, window, lens, (1,) * len(lens))
    plan = ("coop", 1, 0) if split == "coop" else ("coop", 6, 64)
    if split == "coop_split_two_kernels":
        monkeypatch.setattr(attention_mfma, "MERGE_COUNTERS", 0)
    monkeypatch.setattr(attention_mfma, "plan_splits", lambda t, n, m, d=None: plan)
    cu = list(range(len(lens) + 1))
    none = torch.zeros(0, dtype=torch.int32).cuda()
    step = StepContext(num_tokens=len(lens), num_reqs=len(lens), token_ids=none, positions=none, token_req=c["req"],
                       token_seqpos=c["seqpos"], cu_q=torch.tensor(cu, dtype=torch.int32).cuda(),
                       ctx_len=torch.tensor(lens, dtype=torch.int32).cuda(), req_slots=none, groups=[],
                       logit_rows=none, cu_q_host=cu, ctx_len_host=list(lens), max_q_len=1, max_ctx_len=max(lens),
                       dtype=torch.bfloat16)
    handed = []
    real = attention_mfma._fn

    def spy(stem, name, *a, **k):
        fn = real(stem, name, *a, **k)
        if not name.startswith("qvl_attn_mfma_coop"):
            return fn
        return lambda *args: (handed.append((args[5], args[7], args[8])), fn(*args))[1]   # cu_q, tile_req, tile_ct

    monkeypatch.setattr(attention_mfma, "_fn", spy)
    out = attention_mfma.try_attention(c["q"], c["kc"], c["vc"], c["table"], step, nq, window, c["scale"])
    assert handed == [(None, None, None)]
    assert torch.allclose(out.float().cpu(), c["want"], atol=1.5e-2, rtol=2e-2), (out.float().cpu() - c["want"]).abs().max()
    # the same step declared as one that might hold portions: the lists are handed over, the result is the same bits
    step.max_q_len = 2
    handed.clear()
    with_lists = attention_mfma.try_attention(c["q"], c["kc"], c["vc"], c["table"], step, nq, window, c["scale"])
    assert handed and handed[0][0] is not None and torch.equal(with_lists, out)


@pytest.mark.parametrize("nq, nkv, hd, window", [(14, 2, 128, None), (6, 2, 48, 100)])
def test_mixed_step_with_few_long_decoded_tokens(nq, nkv, hd, window, monkeypatch):
    """A prompt portion beside two decoded tokens whose contexts are long: the decoded tokens go to
    the kernel that splits a context among blocks, in a launch of their own, the portion to the
    kernel for many tiles; both write into the same output.  (The limits are set low here so that
    contexts of a few hundred keys count as long.)"""
    from qwen25vl_lite_amd.ops import attention_mfma, kernels
    from qwen25vl_lite_amd.parts import StepContext
    lens, qlens = (333, 300, 17, 280), (40, 1, 17, 1)
    c = _attention_case(torch.bfloat16, nq, nkv, hd, window, lens, qlens)
    monkeypatch.setattr(attention_mfma, "TARGET_BLOCKS", 8)    # the two decoded tokens make 4 blocks, the portions 24 or more
    monkeypatch.setattr(attention_mfma, "MIN_KEYS_PER_SPLIT", 64)
    monkeypatch.setattr(attention_mfma, "SPLIT_FROM_KEYS", 64)
    monkeypatch.setattr(attention_mfma, "ALONE_KEYS", 128)
    cu = [0]
    for ql in qlens:
        cu.append(cu[-1] + ql)
    none = torch.zeros(0, dtype=torch.int32).cuda()
    step = StepContext(num_tokens=cu[-1], num_reqs=len(lens), token_ids=none, positions=none, token_req=c["req"],
                       token_seqpos=c["seqpos"], cu_q=torch.tensor(cu, dtype=torch.int32).cuda(),
                       ctx_len=torch.tensor(lens, dtype=torch.int32).cuda(), req_slots=none, groups=[],
                       logit_rows=none, cu_q_host=cu, ctx_len_host=list(lens), max_q_len=max(qlens),
                       max_ctx_len=max(lens), dtype=torch.bfloat16)
    assert attention_mfma.long_single_tiles(step, nq // nkv, nkv) == (0, 1, 0, 1)
    called = []
    real = attention_mfma._fn
    monkeypatch.setattr(attention_mfma, "_fn", lambda stem, name, *a, **k: (called.append(name), real(stem, name, *a, **k))[1])
    out = attention_mfma.try_attention(c["q"], c["kc"], c["vc"], c["table"], step, nq, window, c["scale"])
    assert "qvl_attn_mfma_coop_merged" in called and "qvl_attn_mfma_block" in called
    err = (out.float().cpu() - c["want"]).abs().max()
    assert torch.allclose(out.float().cpu(), c["want"], atol=1.5e-2, rtol=2e-2), err


@pytest.mark.parametrize("kind", ["narrow", "two_groups", "wide", "planned_longer"])
@pytest.mark.parametrize("nq, nkv, hd, window, ps", [(14, 2, 128, None, 16), (6, 6, 48, None, 48), (3, 3, 128, 1200, 32), (4, 1, 256, None, 16)])
def test_paged_attention_walks_in_parts(nq, nkv, hd, window, ps, kind):
    """Walks long and few enough to be cut: parts that end inside the context, that hold none of some columns' keys, and (a step
    planned for longer contexts than it has, as a captured one is) no key at all.  The counters are back at zero behind every launch, and a second
    one gives the same bits."""
    from types import SimpleNamespace
    import unittest.mock as mock
    from qwen25vl_lite_amd.ops import attention_mfma
    if hd == 256 and kind in ("two_groups", "wide"):
        pytest.skip("built for head sizes up to 128")
    lens, qlens = (1501, 64, 1030), (37, 20, 1)
    c = _attention_case(torch.bfloat16, nq, nkv, hd, window, lens, qlens, ps=ps)
    cu = [0, 37, 57, 58]
    planned = [4096] * 3 if kind == "planned_longer" else list(lens)
    cu_q, ctx_len = (torch.tensor(x, dtype=torch.int32).cuda() for x in (cu, lens))
    step = SimpleNamespace(num_reqs=3, cu_q=cu_q, cu_q_host=cu, ctx_len=ctx_len, ctx_len_host=planned, max_q_len=37,
                           max_ctx_len=max(planned), derived={})
    with mock.patch.object(attention_mfma, "plan_splits", lambda t, n, m, d=None: ("tile", 1, 0)):
        outs = [attention_mfma.try_attention(c["q"], c["kc"], c["vc"], c["table"], step, nq, window, c["scale"],
                                             force_groups=2 if kind == "two_groups" else 1, force_wide=kind == "wide") for _ in range(3)]
    plan = next(v for k, v in step.derived.items() if k[0] == "walks")[3]
    assert plan.partials >= 2
    torch.cuda.synchronize()
    assert int(attention_mfma._work_queue(c["q"].device)[0].abs().sum()) == 0
    for out in outs:
        assert torch.equal(out, outs[0])
        assert torch.allclose(out.float().cpu(), c["want"], atol=1.5e-2, rtol=2e-2), (out.float().cpu() - c["want"]).abs().max()


@pytest.mark.parametrize("known", [True, False])
@pytest.mark.parametrize("nq, nkv, hd, window, ps", [(14, 2, 128, None, 16), (3, 3, 128, 700, 32), (6, 6, 48, 700, 16)])
def test_paged_attention_of_longer_contexts_than_planned(nq, nkv, hd, window, ps, known):
    """Walks cut for shorter contexts than they meet: the last part goes on to the end, and a window that has moved on leaves the first ones
    without a key; and walks that are whole because nobody knows their lengths."""
    from types import SimpleNamespace
    import unittest.mock as mock
    from qwen25vl_lite_amd.ops import attention_mfma
    lens, qlens, planned = (1501, 64, 1030), (37, 20, 1), [1024, 40, 700]
    c = _attention_case(torch.bfloat16, nq, nkv, hd, window, lens, qlens, ps=ps)
    cu = [0, 37, 57, 58]
    cu_q, ctx_len = (torch.tensor(x, dtype=torch.int32).cuda() for x in (cu, lens))
    step = SimpleNamespace(num_reqs=3, cu_q=cu_q, cu_q_host=cu, ctx_len=ctx_len, ctx_len_host=planned, max_q_len=37,
                           max_ctx_len=max(planned), lengths_known=known, derived={})
    with mock.patch.object(attention_mfma, "plan_splits", lambda t, n, m, d=None: ("tile", 1, 0)):
        out = attention_mfma.try_attention(c["q"], c["kc"], c["vc"], c["table"], step, nq, window, c["scale"],
                                           force_groups=1 if known else None)
    plan = next(v for k, v in step.derived.items() if k[0] == "walks")[3]
    assert plan.partials >= 2 if known else plan.partials == 0
    if known and window:
        first = plan.items[(plan.items[:, 0] == 0) & (plan.items[:, 5] >> 16 > 1) & (plan.items[:, 5] & 0xffff == 0)]
        assert len(first) and (first[:, 4] < (lens[0] - qlens[0] - window + 1) >> 5).any()     # a part 0 that has no key any more
    assert torch.allclose(out.float().cpu(), c["want"], atol=1.5e-2, rtol=2e-2), (out.float().cpu() - c["want"]).abs().max()


@pytest.mark.parametrize("nq, nkv, hd, window, ps", [(28, 4, 128, None, 16), (6, 2, 48, 100, 16), (4, 4, 256, 257, 16),
                                                     (5, 1, 16, None, 16), (28, 4, 128, None, 48), (6, 2, 48, 100, 32),
                                                     (4, 4, 256, 257, 64), (4, 2, 32, None, 16), (8, 2, 64, 70, 32),
                                                     (3, 1, 96, None, 16), (6, 3, 112, 200, 48)])
def test_paged_attention_long_portions(nq, nkv, hd, window, ps):
    """Prompt portions long enough for several blocks of several waves per request, next to a
    short portion and a decoded token: the kernel that shares keys through LDS walks the union of
    its waves' ranges, with blocks that some of its waves skip.  Every head size in steps of 16 up to
    128 lays its stages out differently (loads per part, the second half's offset): all of them run."""
    from qwen25vl_lite_amd.ops import attention_mfma, kernels
    from qwen25vl_lite_amd.parts import StepContext
    lens, qlens = (413, 150, 90), (380, 3, 1)
    c = _attention_case(torch.bfloat16, nq, nkv, hd, window, lens, qlens, ps=ps)
    cu = [0]
    for ql in qlens:
        cu.append(cu[-1] + ql)
    none = torch.zeros(0, dtype=torch.int32).cuda()
    step = StepContext(num_tokens=cu[-1], num_reqs=len(lens), token_ids=none, positions=none, token_req=c["req"],
                       token_seqpos=c["seqpos"], cu_q=torch.tensor(cu, dtype=torch.int32).cuda(),
                       ctx_len=torch.tensor(lens, dtype=torch.int32).cuda(), req_slots=none, groups=[],
                       logit_rows=none, cu_q_host=cu, ctx_len_host=list(lens), max_q_len=max(qlens),
                       max_ctx_len=max(lens), dtype=torch.bfloat16)
    import unittest.mock as mock
    for groups in (1, 2) if hd <= 128 else (1,):   # an odd and an even number of key blocks among the walks
        with mock.patch.object(attention_mfma, "plan_splits", lambda t, n, m, d=None: ("tile", 1, 0)):
            out = attention_mfma.try_attention(c["q"], c["kc"], c["vc"], c["table"], step, nq, window, c["scale"],
                                               force_groups=groups, force_wide=False)
        err = (out.float().cpu() - c["want"]).abs().max()
        assert torch.allclose(out.float().cpu(), c["want"], atol=1.5e-2, rtol=2e-2), (groups, err)
    if hd in (128, 48):   # the kind whose waves carry three column tiles (its operands pass through a few registers)
        with mock.patch.object(attention_mfma, "plan_splits", lambda t, n, m, d=None: ("tile", 1, 0)):
            out = attention_mfma.try_attention(c["q"], c["kc"], c["vc"], c["table"], step, nq, window, c["scale"],
                                               force_groups=1, force_wide=True)
        err = (out.float().cpu() - c["want"]).abs().max()
        assert torch.allclose(out.float().cpu(), c["want"], atol=1.5e-2, rtol=2e-2), ("wide", err)
        assert attention_mfma.block_tiles(hd, True) == 12 and attention_mfma.block_tiles(hd) == 8
    # every launch leaves the work-queue counters at zero for the next one
    torch.cuda.synchronize()
    assert int(attention_mfma._work_queue(c["q"].device)[0].abs().sum()) == 0
    assert attention_mfma.block_groups(10, 512, hd) == (2 if hd <= 128 else 1)
    assert attention_mfma.block_groups(513, 512, hd) == 1
    with mock.patch.object(attention_mfma, "plan_splits", lambda t, n, m, d=None: ("tile", 1, 0)), pytest.raises(kernels.KernelError):
        attention_mfma.try_attention(c["q"], c["kc"], c["vc"], c["table"], step, nq, window, c["scale"], force_groups=3)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows, inter", [(7, 353), (5, 352), (70, 18944)])
def test_swiglu(dtype, rows, inter):
    from qwen25vl_lite_amd.ops import kernels
    torch.manual_seed(3)
    x = (torch.randn(rows, 2 * inter) * 3).to(dtype)
    want = torch.nn.functional.silu(x[:, :inter].float()) * x[:, inter:].float()
    out = kernels.swiglu(x.cuda())
    assert torch.allclose(out.float().cpu(), want, **_tol(dtype))
    if inter % 8 == 0:   # the same values with gate and up columns in alternating groups of 8
        g = torch.stack([x[:, :inter].reshape(rows, -1, 8), x[:, inter:].reshape(rows, -1, 8)], dim=2)
        out = kernels.swiglu(g.reshape(rows, 2 * inter).contiguous().cuda(), grouped=True)
        assert torch.allclose(out.float().cpu(), want, **_tol(dtype))


@pytest.mark.parametrize("m, n, k", [(1, 5, 3), (7, 509, 144), (65, 130, 353), (130, 64, 1000)])
def test_gemm_f32_is_exact_and_row_independent(m, n, k):
    from qwen25vl_lite_amd.ops import kernels
    torch.manual_seed(m)
    x, w, b = torch.randn(m, k), torch.randn(n, k), torch.randn(n)
    want = (x.double() @ w.double().T + b.double()).float()
    out = kernels.gemm_f32(x.cuda(), w.cuda(), b.cuda())
    assert torch.allclose(out.cpu(), want, atol=1e-4 * math.sqrt(k), rtol=1e-5)
    # no reduced-precision input format: products of values that bfloat16/tf32 would round
    xe = torch.full((1, 4), 1 + 2 ** -20)
    we = torch.tensor([[1.0, -1.0, 1.0, -1.0 + 2 ** -19]])
    assert kernels.gemm_f32(xe.cuda(), we.cuda()).item() == pytest.approx((xe.double() @ we.double().T).item(), abs=1e-12)
    # a row's result does not depend on what else is in the batch
    alone = kernels.gemm_f32(x[m // 2:m // 2 + 1].contiguous().cuda(), w.cuda(), b.cuda())
    assert torch.equal(alone[0], out[m // 2])


@pytest.mark.parametrize("n, k", [(5, 4), (64, 60), (130, 64), (33, 68), (509, 1000), (2560, 2048), (16390, 132)])
@pytest.mark.parametrize("m", [1, 16, 17, 33, 64, 65, 130])
def test_gemm_f32_tiles_give_the_chains_bits(m, n, k):
    """The matrix-core tiles (rows on 16-byte boundaries) against the plain kernel, which takes any stride: one chain of
    fused multiply-adds an output in either, so the same bits.  Sizes on either side of a tile, of a step of K, and of
    where another shape of blocks is chosen; denormals and wide ranges among the values."""
    from qwen25vl_lite_amd.ops import kernels
    g = torch.Generator(device="cuda").manual_seed(m * n + k)
    x = torch.randn(m, k, device="cuda", generator=g) * torch.exp2(torch.randint(-30, 30, (m, k), device="cuda", generator=g).float())
    w = torch.randn(n, k, device="cuda", generator=g)
    w[::7] *= 1e-38
    b = torch.randn(n, device="cuda", generator=g)
    wide = torch.zeros(m, k + 1, device="cuda")            # rows no multiple of 16 bytes apart: the plain kernel
    wide[:, :k] = x
    for bias in (None, b):
        want = kernels.gemm_f32(wide[:, :k], w, bias)
        assert torch.equal(kernels.gemm_f32(x, w, bias), want)
    out = torch.empty(m, n + 3, device="cuda")[:, :n]
    assert torch.equal(kernels.gemm_f32(x, w, b, out=out), want)


@pytest.mark.parametrize("n, k", [(2048, 11008), (2049, 2308), (4100, 2052), (70, 8200), (17, 2044), (28700, 260)])
@pytest.mark.parametrize("m", [1, 8, 9, 16, 17, 32, 33, 130])
def test_gemm_f32_ranges_of_k(m, n, k):
    """K in several ranges, the last one short and off the steps of 32; one and several tiles a block, outputs on both
    sides of where a block takes 8 or 16, cut and uncut.  Against 64 bits (a run of 32 products and at most 43 + 8 sums on the way: each
    rounds off half of 2^-23 of a partial sum at most, 2^-23 sqrt(91 / 2) of the result's scale as random errors add) and the plain kernel's bits."""
    from qwen25vl_lite_amd.ops import kernels
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x, w = torch.randn(m, k, device="cuda", generator=g), torch.randn(n, k, device="cuda", generator=g)
    b = torch.randn(n, device="cuda", generator=g)
    got = kernels.gemm_f32(x, w, b)
    want = x.double() @ w.double().t() + b.double()
    assert ((got - want).norm() / want.norm()).item() < 2 ** -23 * (91 / 2) ** 0.5
    wide = torch.zeros(m, k + 1, device="cuda")
    wide[:, :k] = x
    assert torch.equal(kernels.gemm_f32(wide[:, :k], w, b), got)


@pytest.mark.parametrize("n, k", [(40005, 64), (33001, 700), (5000, 1000), (4099, 256), (70, 64), (1030, 516), (300, 2052)])
@pytest.mark.parametrize("m", [1, 16, 17, 33, 64, 100, 300])
def test_gemm_f32_of_few_ranges(m, n, k):
    """One to four ranges, so that the waves of a block of few rows have several tiles of outputs; small tiles and large ones, cut
    and uncut, the last ones not full: against 64 bits, with the plain kernel's bits."""
    from qwen25vl_lite_amd.ops import kernels
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x, w = torch.randn(m, k, device="cuda", generator=g), torch.randn(n, k, device="cuda", generator=g)
    b = torch.randn(n, device="cuda", generator=g)
    got = kernels.gemm_f32(x, w, b)
    want = x.double() @ w.double().t() + b.double()
    assert ((got - want).norm() / want.norm()).item() < 2 ** -23 * (91 / 2) ** 0.5       # as for more ranges
    wide = torch.full((m, k + 1), math.nan, device="cuda")
    wide[:, :k] = x
    assert torch.equal(kernels.gemm_f32(wide[:, :k], w, b), got)
    out = torch.full((m, n + 3), 7.0, device="cuda")
    assert torch.equal(kernels.gemm_f32(x, w, b, out=out[:, 1:n + 1]), got) and bool((out[:, 0] == 7).all()) and bool((out[:, n + 1:] == 7).all())


def test_gemm_f32_of_more_rows_than_a_grid_has_places_for_tiles_of_64():
    from qwen25vl_lite_amd.ops import kernels
    m, n, k = 65535 * 64 + 65, 3, 32
    x, w = torch.randn(m, k, device="cuda"), torch.randn(n, k, device="cuda")
    got = kernels.gemm_f32(x, w)
    for at in (0, 65535 * 32, 65535 * 64 - 40, m - 100):
        assert torch.equal(got[at:at + 100], kernels.gemm_f32(x[at:at + 100], w))


@pytest.mark.parametrize("m, n, k", [(1, 509, 144), (8, 300, 200), (16, 17, 8), (9, 100, 8200), (17, 1000, 4104),
                                     (31, 130, 352), (64, 509, 3584), (5, 40, 100), (300, 64, 1000),
                                     (17, 4700, 3584), (32, 300, 3840), (24, 509, 3848), (20, 33, 8),
                                     (30, 4104, 4000), (16, 4104, 4104), (33, 300, 200), (64, 4700, 3584),
                                     (48, 509, 3848), (41, 130, 8200), (64, 3584, 18944), (65, 300, 200)])
def test_linear_bfloat16(m, n, k):
    """Up to 64 rows go through the resident matrix-core kernel (inner sizes in steps of 8): up to 32
    rows always if the inner size fits one pass of a block (4096, or 3840 with 17 to 32 rows), and
    with a longer one while each compute unit has one tile at most; 33 to 64 rows if it fits one pass
    (teams of blocks); the rest through the library; all accumulate in float32."""
    from qwen25vl_lite_amd.ops import skinny
    from qwen25vl_lite_amd.ops.linear import linear
    torch.manual_seed(k)
    x, w = torch.randn(m, k).bfloat16(), (torch.randn(n, k) / math.sqrt(k)).bfloat16()
    b = torch.randn(n)
    want = x.float() @ w.float().T
    units = torch.cuda.get_device_properties(0).multi_processor_count
    assert skinny.takes_resident(m, k, w.cuda()) == (
        k % 8 == 0 and m <= 64 and (k <= 4096 if m > 32 else (k <= (4096 if m <= 16 else 3840) or n <= 16 * units)))
    out32 = linear(x.cuda(), w.cuda(), out_dtype=torch.float32)
    assert out32.dtype == torch.float32 and torch.allclose(out32.cpu(), want, atol=2e-3, rtol=2e-3)
    out16 = linear(x.cuda(), w.cuda())
    assert out16.dtype == torch.bfloat16 and torch.allclose(out16.float().cpu(), want, atol=2e-2, rtol=2e-2)
    outb = linear(x.cuda(), w.cuda(), b.cuda(), out_dtype=torch.float32)
    assert torch.allclose(outb.cpu(), want + b, atol=2e-3, rtol=2e-3)
    # a row's result does not depend on the rows beside it
    if m > 1:
        alone = linear(x[m // 2:m // 2 + 1].contiguous().cuda(), w.cuda(), out_dtype=torch.float32)
        assert torch.allclose(alone[0], out32[m // 2], atol=1e-5, rtol=1e-5)


@pytest.mark.parametrize("m, n, k", [(1, 48, 64), (7, 1000, 3584), (16, 130, 4096), (3, 64, 144),
                                     (17, 1000, 3584), (32, 130, 3840), (29, 64, 144), (24, 48, 4096),
                                     (33, 1000, 3584), (64, 64, 144)])
def test_product_with_the_norm_folded_in(m, n, k):
    """rmsnorm(h) * w formed inside the product equals the norm kernel followed by the product."""
    from qwen25vl_lite_amd.ops import kernels
    from qwen25vl_lite_amd.ops.linear import NormedRows, linear
    torch.manual_seed(n)
    h = (torch.randn(m, k) * 2).cuda()
    g = (1 + 0.1 * torch.randn(k)).cuda()
    w = (torch.randn(n, k) / math.sqrt(k)).bfloat16().cuda()
    fused = linear(NormedRows(h, g, 1e-5, torch.bfloat16), w, out_dtype=torch.float32)
    apart = linear(kernels.add_rmsnorm(h, None, g, 1e-5, torch.bfloat16), w, out_dtype=torch.float32)
    want = plain_rmsnorm(h.cpu(), g.cpu(), 1e-5).bfloat16().float() @ w.float().cpu().T
    assert torch.allclose(fused.cpu(), want, atol=3e-3, rtol=3e-3)
    assert (fused - apart).abs().max() < 0.02 * want.abs().max()   # the same up to a bfloat16 rounding of x here and there
    if m > 32:   # teams of blocks: `linear` leaves these to the library, the kernel itself takes them
        from qwen25vl_lite_amd.ops import skinny
        assert skinny.folds_norm(m, k)
        team = skinny.resident_product(w, h=h, norm_weight=g, eps=1e-5, out_dtype=torch.float32)
        assert torch.allclose(team.cpu(), want, atol=3e-3, rtol=3e-3)
        both = skinny.resident_product(w, x=kernels.add_rmsnorm(h, None, g, 1e-5, torch.bfloat16), out_dtype=torch.float32)
        assert torch.allclose(both.cpu(), want, atol=3e-3, rtol=3e-3)
    # a longer row than one pass of the block holds is computed by the norm's own kernel first
    h2, g2 = torch.randn(2, 4104).cuda(), torch.ones(4104).cuda()
    w2 = (torch.randn(24, 4104) / 64).bfloat16().cuda()
    out = linear(NormedRows(h2, g2, 1e-6, torch.bfloat16), w2, out_dtype=torch.float32)
    assert torch.allclose(out.cpu(), plain_rmsnorm(h2.cpu(), g2.cpu(), 1e-6).bfloat16().float() @ w2.float().cpu().T,
                          atol=3e-3, rtol=3e-3)


@pytest.mark.parametrize("m, n, k", [(1, 144, 352), (8, 3584, 18944), (16, 100, 4104), (24, 144, 352), (40, 144, 352),
                                     (32, 3584, 3584), (17, 100, 3840), (24, 144, 4104), (32, 3584, 18944),
                                     (64, 3584, 18944), (33, 3584, 3584), (57, 100, 4104), (70, 144, 352)])
def test_product_added_into_the_residual(m, n, k):
    from qwen25vl_lite_amd.ops.linear import linear_into
    torch.manual_seed(k)
    x = torch.randn(m, k).bfloat16().cuda()
    w = (torch.randn(n, k) / math.sqrt(k)).bfloat16().cuda()
    h = torch.randn(m, n).cuda()
    want = h.cpu() + x.float().cpu() @ w.float().cpu().T
    left = linear_into(h, x, w)
    if m <= 16 and k <= 4096:      # one block carries the rows for the whole inner size: added in place
        assert left is None and torch.allclose(h.cpu(), want, atol=3e-3, rtol=3e-3)
    elif m <= 64:   # the split kernel: slabs of partial sums for the next norm to add
        assert left.dtype == torch.float32 and left.dim() == 3 and tuple(left.shape[1:]) == (m, n)
        assert torch.allclose(h.cpu() + left.sum(0).cpu(), want, atol=3e-3, rtol=3e-3)
    else:   # the library's product comes back in bfloat16 for the next norm to add
        assert left is not None and left.dtype == torch.bfloat16 and left.dim() == 2
        assert torch.allclose(h.cpu() + left.float().cpu(), want, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m, inter, k", [(1, 352, 144), (8, 18944, 3584), (16, 40, 4104), (50, 352, 144),
                                         (4, 2072, 64), (3, 5136, 72), (2, 8 * 320, 40),
                                         (32, 18944, 3584), (17, 2072, 64), (25, 5136, 72), (64, 18944, 3584),
                                         (33, 2072, 64), (47, 5136, 72), (70, 352, 144)])
def test_gate_up_product_with_the_activation_folded_in(dtype, m, inter, k):
    """Grouped gate | up rows: few bfloat16 rows get silu(gate) * up from the product's own kernel,
    everything else from the product followed by the activation kernel on the grouped columns."""
    from qwen25vl_lite_amd.ops.linear import gate_up_swiglu
    torch.manual_seed(inter)
    x = torch.randn(m, k).to(dtype)
    gate = (torch.randn(inter, k) / math.sqrt(k)).to(dtype)
    up = (torch.randn(inter, k) / math.sqrt(k)).to(dtype)
    grouped = torch.stack([gate.view(-1, 8, k), up.view(-1, 8, k)], dim=1).reshape(2 * inter, k).contiguous()
    out = gate_up_swiglu(x.cuda(), grouped.cuda(), True)
    want = torch.nn.functional.silu(x.float() @ gate.float().T) * (x.float() @ up.float().T)
    assert out.shape == (m, inter) and out.dtype == dtype
    tol = dict(atol=1e-4, rtol=1e-4) if dtype == torch.float32 else dict(atol=2e-2, rtol=2e-2)
    assert torch.allclose(out.float().cpu(), want, **tol)
    plain = gate_up_swiglu(x.cuda(), torch.cat([gate, up]).cuda(), False)
    assert torch.allclose(plain.float().cpu(), want, **tol)


@pytest.mark.parametrize("m, n, k", [(64, 3584, 18944), (17, 509, 352), (33, 130, 200), (48, 1000, 3584), (40, 144, 352),
                                     (64, 37, 8), (25, 4700, 1248), (57, 300, 1256), (1, 3584, 18944), (8, 2048, 11008),
                                     (16, 37, 4104), (3, 5000, 2056), (49, 8, 2048 * 300 + 8), (4, 512, 29568), (33, 260, 29568)])
def test_split_product_and_the_norm_that_adds_its_slabs(m, n, k):
    """Up to 64 rows against a weight cut along its inner size: the slabs of partial sums add up to
    the product (inner sizes that are no multiple of 32, row counts that fill no tile, more chunks
    than compute units refused), twice the same bits; and the norm kernel that takes the slabs as
    its addend gives what it gives for their sum."""
    from qwen25vl_lite_amd.ops import kernels, skinny
    torch.manual_seed(n + k)
    w = (torch.randn(n, k) / math.sqrt(k)).bfloat16()
    x = torch.randn(m, k).bfloat16()
    want = x.float() @ w.float().T
    if k > 2048 * 256:
        assert not skinny.takes_split(m, k, w.cuda())
        with pytest.raises(ValueError):
            skinny.split_product(w.cuda(), x.cuda())
        return
    assert skinny.takes_split(m, k, w.cuda()) and not skinny.takes_split(65, k, w.cuda())
    slabs = skinny.split_product(w.cuda(), x.cuda())
    assert slabs.dtype == torch.float32 and slabs.dim() == 3 and tuple(slabs.shape[1:]) == (m, n)
    assert torch.allclose(slabs.sum(0).cpu(), want, atol=3e-3, rtol=3e-3), (slabs.sum(0).cpu() - want).abs().max()
    assert torch.equal(slabs, skinny.split_product(w.cuda(), x.cuda()))
    if n % 4 == 0:
        h = torch.randn(m, n).cuda()
        g = (1 + 0.1 * torch.randn(n)).cuda()
        h1, h2 = h.clone(), h.clone()
        a = kernels.add_rmsnorm(h1, slabs, g, 1e-6, torch.bfloat16)
        total = slabs[0].clone()
        for c in range(1, slabs.shape[0]):
            total += slabs[c]
        b = kernels.add_rmsnorm(h2, total, g, 1e-6, torch.bfloat16)
        assert torch.equal(h1, h2), "the slabs are added in their order"
        # (the two kernels add the squares up in different orders: the scale may differ in its last bit)
        assert torch.allclose(a.float(), b.float(), atol=1e-2, rtol=1e-2)
        rows = torch.tensor([m - 1, 0], dtype=torch.int32).cuda()
        h3 = h.clone()
        c3 = kernels.add_rmsnorm(h3, slabs, g, 1e-6, torch.float32, rows=rows)
        assert torch.equal(h3, h) and torch.allclose(c3, kernels.add_rmsnorm(h.clone(), total, g, 1e-6, torch.float32)[[m - 1, 0]])


def test_few_row_products_at_random_sizes():
    """The resident kernel (both builds: inner sizes up to and beyond 2,048) and the split kernel at
    sizes drawn at random: any row count up to 64, widths that fill no tile, inner sizes in steps of 8
    on either side of a pass, of a chunk and of a build; every one against the float32 product."""
    import random
    from qwen25vl_lite_amd.ops import skinny
    from qwen25vl_lite_amd.ops.linear import linear, linear_into
    rng = random.Random(5)
    edges = [8, 120, 128, 136, 1016, 1024, 2040, 2048, 2056, 3832, 3840, 3848, 4088, 4096, 4104, 6144, 8200]
    for case in range(48):
        m = rng.choice([1, 2, 7, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64])
        n = rng.choice([1, 5, 15, 16, 17, 100, 255, 256, 257, 1000])
        k = rng.choice(edges) if case % 2 else 8 * rng.randint(1, 700)
        torch.manual_seed(case)
        x = torch.randn(m, k).bfloat16().cuda()
        w = (torch.randn(n, k) / math.sqrt(k)).bfloat16().cuda()
        want = x.float() @ w.float().T
        got = linear(x, w, out_dtype=torch.float32)
        assert torch.allclose(got, want, atol=5e-3, rtol=5e-3), (m, n, k, (got - want).abs().max().item())
        slabs = skinny.split_product(w, x)
        assert torch.allclose(slabs.sum(0), want, atol=5e-3, rtol=5e-3), (m, n, k, (slabs.sum(0) - want).abs().max().item())
        h = torch.randn(m, n).cuda()
        before = h.clone()
        left = linear_into(h, x, w)
        total = h if left is None else h + (left.sum(0) if left.dim() == 3 else left.float())
        assert torch.allclose(total, before + want, atol=2e-2, rtol=2e-2), (m, n, k)


@pytest.mark.parametrize("m", [1, 16, 17, 33, 64])
@pytest.mark.parametrize("k", [8, 136, 1016, 2040, 2056, 3832])
def test_few_row_products_read_nothing_beside_the_inner_size(m, k):
    """The weight comes through LDS in units of 128 columns: with NaN behind the inner size in every row of both operands,
    the last unit's columns beyond it must not be part of a sum, with the rows as they are, with their norm
    formed inside, and over ranges of the inner size.  Each sum of k exact products is within k roundings of its terms."""
    from qwen25vl_lite_amd.ops import kernels, skinny
    torch.manual_seed(m + k)
    n = 300
    nan = float("nan")
    wide_w, wide_x, wide_h = (torch.full((r, k + 128), nan, device="cuda") for r in (n, m, m))
    wide_w, wide_x = wide_w.bfloat16(), wide_x.bfloat16()
    w, x, h = wide_w[:, :k], wide_x[:, :k], wide_h[:, :k]
    w.copy_(torch.randn(n, k) / math.sqrt(k))
    x.copy_(torch.randn(m, k))
    h.copy_(torch.randn(m, k))
    g = (1 + 0.1 * torch.randn(k)).cuda()

    def near(got, a, slack=0.0):
        a, b = a.double().cpu(), w.double().cpu()
        err = (got.double().cpu() - a @ b.T).abs()
        assert bool((err <= (k * 2.0 ** -24 + slack) * (a.abs() @ b.abs().T) + 1e-30).all()), err.max()

    near(skinny.resident_product(w, x=x), x)
    near(skinny.split_product(w, x).sum(0), x)
    if skinny.folds_norm(m, k):
        # (a normed value may be rounded to bfloat16's other neighbour: the statistics are added up in another order)
        near(skinny.resident_product(w, h=h, norm_weight=g, eps=1e-6), kernels.add_rmsnorm(h.contiguous(), None, g, 1e-6, torch.bfloat16),
             2.0 ** -8)


def _off(got, x, w):
    """Error of a product against 64 bits, 2-norm over 2-norm."""
    want = x.double() @ w.double().T
    return float((got.double() - want).norm() / want.norm())


@pytest.mark.parametrize("m", [1, 8, 16, 24])
@pytest.mark.parametrize("k", [896, 1024, 1536, 2048, 3584, 4096])
def test_float32_sums_of_the_resident_kernel(m, k):
    """As below: chains of at most 8 products of 32 values, which the instruction adds in two halves, a join of the two halves of
    a wave's columns and one sum for each of up to 8 waves: sqrt(8 + 1 / 2 + 4) of 2^-24 / sqrt(3) at most."""
    from qwen25vl_lite_amd.ops import skinny
    torch.manual_seed(m + k)
    x = torch.randn(m, k, device="cuda").bfloat16()
    w = (torch.randn(2048, k, device="cuda") / math.sqrt(k)).bfloat16()
    bound = 2.0 ** -24 / math.sqrt(3.0) * math.sqrt(12.5)
    assert _off(skinny.resident_product(w, x=x), x, w) < bound
    if m <= skinny.KEPT_SPLIT_ROWS:
        assert _off(skinny.split_product(w, x).double().sum(0), x, w) < bound


@pytest.mark.parametrize("m", [1, 16, 19, 40, 64])
@pytest.mark.parametrize("k", [1024, 3584, 8192])
def test_float32_sums_of_the_streaming_kernel(m, k):
    """A chain of additions is off by a random walk: each rounds off up to half a unit of 24 bits (2^-24 / sqrt(3) on
    average) of a sum that grows evenly, sqrt(n / 2) of them in the end.  Sums are formed of chains of 16 at most, two levels of
    joins and a join for every 512 values: no more than sqrt(8 + 2 + k / 1024) of them."""
    from qwen25vl_lite_amd.ops import rows, skinny
    torch.manual_seed(m + k)
    x = torch.randn(m, k, device="cuda").bfloat16()
    w = (torch.randn(2048, k, device="cuda") / math.sqrt(k)).bfloat16()
    bound = 2.0 ** -24 / math.sqrt(3.0) * math.sqrt(10 + k / 1024)
    assert _off(rows.rows_product(x, w, torch.float32), x, w) < bound
    if m > skinny.KEPT_SPLIT_ROWS:
        slabs = skinny.split_product(w, x)
        assert _off(slabs.double().sum(0), x, w) < bound


@pytest.mark.parametrize("m", [1, 19, 32, 33, 64])
@pytest.mark.parametrize("n, k", [(16, 8), (16400, 136), (37888, 72), (59136, 64), (81920, 200), (152064, 136), (36912, 2056)])
def test_rows_against_many_outputs(m, n, k):
    """The kernel for up to 64 rows and many outputs: two, three and four fetches of the weight's rows a wave, one round of tiles
    and several, inner sizes that end inside a step, NaN behind the inner size in every row, an odd row stride of the
    result; each sum of k exact products is within k roundings of its terms, a stored bfloat16 half a unit in its last place
    further; gated values against the same activation of the float32 products."""
    from qwen25vl_lite_amd.ops import rows
    torch.manual_seed(m + n)
    wide_w = torch.full((n, k + 64), float("nan"), device="cuda").bfloat16()
    wide_x = torch.full((m, k + 64), float("nan"), device="cuda").bfloat16()
    w, x = wide_w[:, :k], wide_x[:, :k]
    w.copy_(torch.randn(n, k, device="cuda") / math.sqrt(k))
    x.copy_(torch.randn(m, k, device="cuda"))
    want = x.double() @ w.double().T
    bound = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) + 1e-30
    sums = rows.rows_product(x, w, torch.float32)
    assert bool(((sums.double() - want).abs() <= bound).all())
    for wider in (0, 1, 2):
        out = torch.full((m, n + wider), 7.0, device="cuda").bfloat16()
        rows.rows_product(x, w, out=out[:, :n])
        assert bool(((out[:, :n].double() - want).abs() <= bound + 2.0 ** -8 * want.abs()).all())
        assert bool((out[:, n:] == 7.0).all())
    pairs = want.view(m, n // 16, 2, 8)
    for act, fn in (("silu", torch.nn.functional.silu), ("gelu_tanh", lambda t: torch.nn.functional.gelu(t, approximate="tanh"))):
        got = rows.rows_swiglu(x, w, act).double()
        ref = (fn(pairs[:, :, 0]) * pairs[:, :, 1]).reshape(m, n // 2)
        # both factors' sums within their bounds (an activation's slope is below 1.13), float32 rounding of the activation, one to bfloat16
        b = bound.view(m, n // 16, 2, 8)
        slack = (1.13 * b[:, :, 0] * (pairs[:, :, 1].abs() + b[:, :, 1]) + fn(pairs[:, :, 0]).abs() * b[:, :, 1]).reshape(m, n // 2)
        assert bool(((got - ref).abs() <= slack + (2.0 ** -8 + 1e-5) * ref.abs() + 1e-5 * pairs[:, :, 1].abs().reshape(m, n // 2)).all())
    # all gate rows, then the up rows; with clamps the values are at most 1.5 and 2.5, the slopes 1.13 and 1
    got = rows.rows_gated(x, w, 1.25, 1.5, 1.0).double()
    g, u = want[:, :n // 2].clamp(max=1.5), want[:, n // 2:].clamp(-1.5, 1.5)
    ref = g * torch.sigmoid(1.25 * g) * (u + 1.0)
    slack = 1.13 * 2.5 * bound[:, :n // 2] + 1.5 * bound[:, n // 2:]
    assert bool(((got - ref).abs() <= slack + (2.0 ** -8 + 1e-6) * ref.abs() + 2e-6).all())


@pytest.mark.parametrize("e, top, groups, keep, score", [(1, 1, 1, 1, "softmax"), (32, 6, 1, 1, "softmax"), (64, 8, 1, 1, "sigmoid"),
                                                         (65, 64, 1, 1, "sigmoid"), (512, 8, 1, 1, "softmax"), (72, 5, 8, 3, "sigmoid")])
def test_routes_listed_by_expert(e, top, groups, keep, score):
    """Rows for one wave and for several of a block, and one more than it takes; logits from a few values, so that most choices are
    among equals and the lower index has to win; the listing holds every pair once, under its expert."""
    from qwen25vl_lite_amd.ops import moe
    for n in (1, 16, 17, 64, 65, 200):
        torch.manual_seed(n)
        z = torch.randint(0, 5, (n, e), device="cuda").float()
        ids, wts, order, offsets = moe.route_sorted(z, top, groups, keep, 1.5, score)
        s = torch.softmax(z.double(), -1) if score == "softmax" else torch.sigmoid(z.double())
        if groups > 1:
            members = s.view(n, groups, e // groups)
            best = members.topk(2, -1).values.sum(-1)
            rank = (best[:, None, :] > best[:, :, None]).sum(-1) + ((best[:, None, :] == best[:, :, None])
                                                                      & (torch.arange(groups, device="cuda")[None, None] < torch.arange(groups, device="cuda")[None, :, None])).sum(-1)
            members = members.masked_fill((rank >= keep)[:, :, None], -1.0)
            s = members.reshape(n, e)
        # the lower index first among equals: a stable sort downwards
        want = torch.sort(s, dim=-1, descending=True, stable=True)
        assert torch.equal(ids.long(), want.indices[:, :top]), n
        w = want.values[:, :top]
        assert torch.allclose(wts.double(), 1.5 * w / w.sum(-1, keepdim=True), rtol=1e-5, atol=0)
        flat = ids.view(-1).long()
        assert torch.equal(offsets.long(), torch.cat([torch.zeros(1, device="cuda").long(), torch.bincount(flat, minlength=e).cumsum(0)]))
        assert torch.equal(order.long().sort().values, torch.arange(n * top, device="cuda"))
        assert torch.equal(flat[order.long()], flat.sort().values)
        again = moe.route(z, top, groups, keep, 1.5, score)
        assert torch.equal(again[0], ids) and torch.equal(again[1], wts)


@pytest.mark.parametrize("e, top, groups, keep", [(1, 1, 1, 1), (70, 64, 1, 1), (512, 8, 8, 4)])
def test_routes_listed_on_both_sides_of_one_launch(e, top, groups, keep):
    from qwen25vl_lite_amd.ops import moe
    for n in (1, 7, 8, 9, 16):
        torch.manual_seed(n)
        z = torch.randn(n, e, device="cuda")
        ids, wts, order, offsets = moe.route_sorted(z, top, groups, keep, 1.5)
        again = moe.route(z, top, groups, keep, 1.5)
        assert torch.equal(again[0], ids) and torch.equal(again[1], wts)
        flat = ids.view(-1).long()
        assert torch.equal(offsets.long(), torch.cat([torch.zeros(1, device="cuda").long(), torch.bincount(flat, minlength=e).cumsum(0)]))
        assert torch.equal(order.long().sort().values, torch.arange(n * top, device="cuda")) and torch.equal(flat[order.long()], flat.sort().values)


@pytest.mark.parametrize("e, r, k, pairs", [(3, 40, 72, "one"), (8, 300, 200, "uneven"), (70, 129, 64, "uneven"), (4, 2368, 136, "all on one"),
                                            (200, 1, 8, "uneven"), (32, 520, 2056, "few")])
def test_experts_with_few_pairs(e, r, k, pairs):
    """The experts' products of a decode step: experts with no pair, with one and with more than the 32 of a tile, rows and
    inner sizes that fill no tile and no step, NaN beside the rows of x, more experts than lanes; plain, squared and
    gated, both output types.  A sum of k exact products is within k roundings of its terms."""
    from qwen25vl_lite_amd.ops import moe
    torch.manual_seed(e + r)
    top, n = 2, {"one": 1, "uneven": 45, "all on one": 20, "few": 8}[pairs]
    ids = torch.randint(0, e, (n, top), dtype=torch.int32, device="cuda")
    if pairs == "uneven":
        ids[:, 0] = e // 2
    elif pairs == "all on one":
        ids[:] = 2
    order, offsets = moe.sort_pairs(ids, e)
    x = torch.full((n, k + 64), float("nan"), device="cuda").bfloat16()[:, :k]
    x.copy_(torch.randn(n, k, device="cuda"))
    w = (torch.randn(e, 2 * r, k, device="cuda") / math.sqrt(k)).bfloat16()
    flat = ids.view(-1).long()
    xs, ws = x.double().repeat_interleave(top, 0), w.double()[flat]
    want = torch.einsum("pk,prk->pr", xs, ws)
    bound = k * 2.0 ** -24 * torch.einsum("pk,prk->pr", xs.abs(), ws.abs()) + 1e-30
    got = moe.expert_products(x, w, order, offsets, n * top, top, torch.float32)
    assert bool(((got.double() - want).abs() <= bound).all())
    room = torch.full((n * top, 2 * r + 3), 7.0, device="cuda").bfloat16()
    moe.expert_products(x, w, order, offsets, n * top, top, torch.bfloat16, act="relu2", out=room[:, :2 * r])
    ref = want.clamp(min=0) ** 2
    slack = (2 * want.abs() + bound) * bound
    assert bool(((room[:, :2 * r].double() - ref).abs() <= slack + (2.0 ** -8 + 1e-6) * ref).all()) and bool((room[:, 2 * r:] == 7.0).all())
    g, u = want[:, :r].clamp(max=1.5), want[:, r:].clamp(-1.5, 1.5)
    ref = g * torch.sigmoid(1.25 * g) * (u + 1.0)
    # slopes: of g sigmoid(1.25 g) below 1.13, of u one; values |u + 1| <= 2.5, |g sigmoid| <= 1.5 above and 0.3 below
    slack = 1.13 * 2.5 * bound[:, :r] + 1.5 * bound[:, r:]
    for dtype, last in ((torch.float32, 0.0), (torch.bfloat16, 2.0 ** -8)):
        got = moe.expert_products(x, w, order, offsets, n * top, top, dtype, gated=(1.25, 1.5, 1.0)).double()
        assert bool(((got - ref).abs() <= slack + (last + 1e-6) * ref.abs() + 2e-6).all())


@pytest.mark.parametrize("e, r, k, per", [(2, 300, 160, 255), (2, 300, 160, 257), (3, 128, 96, 700), (1, 129, 64, 256), (5, 8, 32, 300)])
def test_experts_with_many_pairs(e, r, k, per):
    """On both sides of where tiles of 256 pairs begin; experts whose pairs fill no tile, outputs that fill none, one expert without
    pairs.  A sum of k exact products is within k roundings of its terms."""
    from qwen25vl_lite_amd.ops import moe
    torch.manual_seed(e + per)
    n, top = per * e // 2 + (per * e) % 2, 2
    ids = torch.randint(0, max(1, e - 1), (n, top), dtype=torch.int32, device="cuda")
    order, offsets = moe.sort_pairs(ids, e)
    x = torch.randn(n, k, device="cuda").bfloat16()
    w = (torch.randn(e, 2 * r, k, device="cuda") / math.sqrt(k)).bfloat16()
    flat = ids.view(-1).long()
    want = torch.zeros(n * top, 2 * r, dtype=torch.float64, device="cuda")
    bound = torch.zeros_like(want)
    for i in range(e):
        at = (flat == i).nonzero()[:, 0]
        want[at] = x[at // top].double() @ w[i].double().t()
        bound[at] = k * 2.0 ** -24 * (x[at // top].double().abs() @ w[i].double().abs().t()) + 1e-30
    got = moe.expert_products(x, w, order, offsets, n * top, top, torch.float32)
    assert bool(((got.double() - want).abs() <= bound).all())
    g, u = want[:, :r].clamp(max=1.5), want[:, r:].clamp(-1.5, 1.5)
    ref = g * torch.sigmoid(1.25 * g) * (u + 1.0)
    slack = 1.13 * 2.5 * bound[:, :r] + 1.5 * bound[:, r:]
    got = moe.expert_products(x, w, order, offsets, n * top, top, torch.bfloat16, gated=(1.25, 1.5, 1.0)).double()
    assert bool(((got - ref).abs() <= slack + (2.0 ** -8 + 1e-6) * ref.abs() + 2e-6).all())


@pytest.mark.parametrize("e, r, k, per", [(3, 1029, 96, 700), (7, 1030, 160, 260), (2, 1033, 32, 1030)])
def test_experts_in_tiles_of_256_pairs(e, r, k, per):
    """Sizes at which these are taken for both products: experts whose pairs fill no tile, outputs off steps of four, a last step of
    half its size."""
    from qwen25vl_lite_amd.ops import kernels
    wide = kernels._fn("moe", "qvl_moe_wide_pairs", [kernels._c_int] * 6)
    pairs = per * e + (per * e) % 2
    assert wide(pairs, e, 2 * r, k, 0, kernels.compute_units("cuda:0")) and wide(pairs, e, r, k, 1, kernels.compute_units("cuda:0"))
    test_experts_with_many_pairs(e, r, k, per)


@pytest.mark.parametrize("m", [1, 16, 32])
def test_rows_of_gate_and_up_that_form_no_groups_keep_the_norm_in_the_product(m, monkeypatch):
    """An inner size of the feed-forward off steps of 8: the product forms the norm of a decode step's rows itself, without a
    kernel in front of it.  The normed rows and the product are rounded to bfloat16, the activation's factors likewise."""
    from qwen25vl_lite_amd.ops import linear as products
    torch.manual_seed(m)
    h = torch.randn(m, 512, device="cuda")
    gain = torch.rand(512, device="cuda") + 0.5
    w = (torch.randn(2 * 1003, 512, device="cuda") / math.sqrt(512)).bfloat16()
    normed = products.NormedRows(h, gain, 1e-6, torch.bfloat16)
    x = normed.materialize().double()

    def apart(self):
        raise AssertionError("the norm ran apart from the product")
    monkeypatch.setattr(products.NormedRows, "materialize", apart)
    got = products.gate_up_swiglu(normed, w, grouped=False).double()
    both = x @ w.double().T
    # each normed value may be the neighbouring bfloat16; float32 sums of 512 products; the product's rounding to bfloat16
    off = (2.0 ** -8 + 512 * 2.0 ** -24) * (x.abs() @ w.double().abs().T) + 2.0 ** -8 * both.abs()
    g, u = both[:, :1003], both[:, 1003:]
    ref = torch.nn.functional.silu(g) * u
    # (the activation's slope is below 1.13)
    slack = 1.13 * off[:, :1003] * (u.abs() + off[:, 1003:]) + torch.nn.functional.silu(g).abs() * off[:, 1003:]
    assert bool(((got - ref).abs() <= slack + 2.0 ** -8 * (ref.abs() + slack)).all())


def test_no_cpu_path():
    from qwen25vl_lite_amd.ops import kernels
    from qwen25vl_lite_amd.ops.linear import linear
    with pytest.raises(kernels.KernelError):
        kernels.swiglu(torch.zeros(2, 4))
    with pytest.raises(kernels.KernelError):
        linear(torch.zeros(2, 4), torch.zeros(3, 4))
    with pytest.raises(kernels.KernelError):
        kernels.swiglu(torch.zeros(2, 4, dtype=torch.float16).cuda())


@pytest.mark.parametrize("ps", [16, 32, 48])
@pytest.mark.parametrize("m, nq, nkv, hd, k, bias, lazy", [(1, 4, 2, 16, 64, True, False), (8, 28, 4, 128, 3584, True, True),
                                                         (16, 6, 3, 48, 136, False, True), (5, 3, 0, 80, 104, True, False),
                                                         (32, 28, 4, 128, 3584, True, True), (17, 6, 3, 48, 136, False, True),
                                                         (27, 4, 2, 16, 64, True, False), (64, 28, 4, 128, 3584, True, False),
                                                         (33, 6, 3, 48, 136, False, False), (50, 4, 2, 16, 64, True, False)])
def test_projection_with_rotation_and_cache_write_folded_in(m, nq, nkv, hd, k, bias, lazy, ps):
    """The stacked q | k | v projection of a few rows that rotates and stores inside the product's
    kernel equals the product followed by the rotation kernel: queries, and every slot of the
    cache (the slots of other tokens keep their stale values)."""
    from qwen25vl_lite_amd.ops import kernels, skinny
    from qwen25vl_lite_amd.ops.linear import linear
    torch.manual_seed(hd + m)
    pages = 7
    n_out = (nq + 2 * nkv) * hd
    w = (torch.randn(n_out, k) / math.sqrt(k)).bfloat16().cuda()
    b = torch.randn(n_out).cuda() if bias else None
    h = (torch.randn(m, k) * 2).cuda()
    g = (1 + 0.1 * torch.randn(k)).cuda()
    x = kernels.add_rmsnorm(h, None, g, 1e-6, torch.bfloat16)
    half = hd // 2
    inv_freq = (1.0 / (10000.0 ** (torch.arange(0, hd, 2, dtype=torch.float32) / hd))).cuda()
    freq_row = (torch.arange(half) % 3).int().cuda()
    if half > 3:
        freq_row[3] = -1                        # a frequency that is not rotated
    pos = torch.randint(0, 40000, (3, m), dtype=torch.int32).cuda()
    slots = torch.randperm(pages * ps)[:m].int().cuda()
    if m > 2:
        slots[1] = -1                           # a token without a slot writes nothing
    kc0 = torch.randn(pages, max(nkv, 1), ps, hd).bfloat16().cuda()
    vc0 = torch.randn(pages, max(nkv, 1), hd, ps).bfloat16().cuda()
    kc_a, vc_a, kc_b, vc_b = kc0.clone(), vc0.clone(), kc0.clone(), vc0.clone()
    qkv = linear(x, w, out_dtype=torch.float32)
    q_a = kernels.rope_kv_write(qkv, b, pos, inv_freq, freq_row, slots if nkv else None, kc_a if nkv else None,
                                vc_a if nkv else None, nq, nkv, hd, ps, out_dtype=torch.bfloat16)
    assert skinny.takes_qkv_rope(m, k, w, hd, half, torch.bfloat16, norm=lazy)
    cs = kernels.rope_table(pos, inv_freq, freq_row, m)
    src = dict(h=h, norm_weight=g, eps=1e-6) if lazy else dict(x=x)
    q_b = skinny.qkv_rope_product(w, cs, bias=b, slots=slots if nkv else None, k_cache=kc_b if nkv else None,
                                  v_cache=vc_b if nkv else None, num_q_heads=nq, num_kv_heads=nkv, head_dim=hd,
                                  page_size=ps, **src)
    tol = dict(atol=2e-2, rtol=2e-2)           # one bfloat16 rounding of values of a few units
    assert torch.allclose(q_b.float(), q_a.float(), **tol), (q_b.float() - q_a.float()).abs().max()
    assert torch.allclose(kc_b.float(), kc_a.float(), **tol) and torch.allclose(vc_b.float(), vc_a.float(), **tol)
    if nkv:   # something was written, and only in the tokens' slots
        assert not torch.equal(kc_b, kc0) and not torch.equal(vc_b, vc0)
        touched = (kc_b != kc0).any(dim=3).any(dim=1).flatten().nonzero().flatten().tolist()
        assert set(touched) <= set(s for s in slots.tolist() if s >= 0)
    # And against the plain formulas themselves (not another path of the engine): the frequencies'
    # rows laid out by sections, the product in float32 on the host, the reference's rotation.
    sections = (half - 2 * (half // 3), half // 3, half // 3)
    rows = torch.tensor(sum(([r] * c for r, c in enumerate(sections)), []), dtype=torch.int32).cuda()
    kc_c, vc_c = kc0.clone(), vc0.clone()
    q_c = skinny.qkv_rope_product(w, kernels.rope_table(pos, inv_freq, rows, m), bias=b, slots=slots if nkv else None,
                                  k_cache=kc_c if nkv else None, v_cache=vc_c if nkv else None, num_q_heads=nq,
                                  num_kv_heads=nkv, head_dim=hd, page_size=ps, **src)
    xb = x.float().cpu() @ w.float().cpu().T + (b.cpu() if bias else 0.0)
    qs, ks, vs = xb.split([nq * hd, nkv * hd, nkv * hd], dim=1)
    cos, sin = plain_mrope_cos_sin(pos.cpu(), inv_freq.cpu())
    heads = lambda t, n: t.reshape(m, n, hd).transpose(0, 1)
    qr, kr = plain_apply_mrope(heads(qs, nq), heads(ks, nkv) if nkv else heads(qs, nq), cos, sin, sections)
    plain_tol = dict(atol=3e-2, rtol=2e-2)     # the norm's output and the result each rounded to bfloat16 once
    assert torch.allclose(q_c.float().cpu().view(m, nq, hd), qr.transpose(0, 1), **plain_tol)
    if nkv:
        kflat = kc_c.float().cpu().permute(0, 2, 1, 3).reshape(pages * ps, nkv, hd)
        vflat = vc_c.float().cpu().permute(0, 3, 1, 2).reshape(pages * ps, nkv, hd)
        live = (slots >= 0).cpu()
        at = slots.cpu().long()[live]
        assert torch.allclose(kflat[at], kr.transpose(0, 1)[live], **plain_tol)
        assert torch.allclose(vflat[at], vs.view(m, nkv, hd)[live], **plain_tol)
    # a head size whose rotation the kernel does not take, or a cache of another type, is refused
    assert not skinny.takes_qkv_rope(m, k, w, 24, 12, torch.bfloat16)
    assert not skinny.takes_qkv_rope(m, k, w, hd, half - 1, torch.bfloat16)
    assert not skinny.takes_qkv_rope(m, k, w, hd, half, torch.float32)


@pytest.mark.parametrize("shape", [0, 1, 2, 3, -1])
@pytest.mark.parametrize("m, n, k", [(65, 16, 32), (128, 256, 64), (129, 272, 96), (256, 500, 544), (257, 1040, 160), (300, 48, 2368)])
def test_tiled_product(m, n, k, shape):
    """The tiled kernel in every tile shape: rows and outputs at and beyond a tile's edges, inner sizes that end with
    half a step, rows further apart than they are wide; stored as bfloat16 and float32, squared, gated both ways."""
    from qwen25vl_lite_amd.ops import tile
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k + 8, device="cuda", generator=g).bfloat16()[:, :k]
    w = (torch.randn(n, k + 16, device="cuda", generator=g) * 2 / k ** 0.5).bfloat16()[:, :k]
    want = x.float() @ w.float().T
    # float32 sums of k products of values about 1 and 2 / sqrt(k) in another order; bfloat16 keeps 8 bits
    exact, rounded = dict(atol=2e-5, rtol=1e-4), dict(atol=1e-2, rtol=1e-2)
    assert torch.allclose(tile.tile_product(x, w, torch.float32, shape=shape), want, **exact)
    out = torch.empty(m, n + 24, dtype=torch.bfloat16, device="cuda")[:, 8:8 + n]
    out[:] = 7.0
    tile.tile_product(x, w, out=out, shape=shape)
    assert torch.allclose(out.float(), want, **rounded)
    assert torch.allclose(tile.tile_product(x, w, relu2=True, shape=shape).float(), want.clamp(min=0) ** 2, atol=2e-2, rtol=2e-2)
    both = want.view(m, n // 16, 2, 8) if n % 16 == 0 else None
    if both is not None:
        for act, fn in (("silu", torch.nn.functional.silu), ("gelu_tanh", lambda z: torch.nn.functional.gelu(z, approximate="tanh"))):
            ref = (fn(both[:, :, 0]) * both[:, :, 1]).reshape(m, n // 2)
            assert torch.allclose(tile.tile_swiglu(x, w, act, shape=shape).float(), ref, atol=2e-2, rtol=2e-2)
    gate, up = want[:, :n // 2].clamp(max=1.5), want[:, n // 2:].clamp(-1.5, 1.5)
    ref = gate * torch.sigmoid(1.702 * gate) * (up + 1.0)
    assert torch.allclose(tile.tile_gated(x, w, 1.702, 1.5, 1.0, shape=shape).float(), ref, atol=2e-2, rtol=2e-2)
    gate, up = want[:, :n // 2], want[:, n // 2:]
    assert torch.allclose(tile.tile_gated(x, w, 1.0, None, 0.0, shape=shape).float(), gate * torch.sigmoid(gate) * up, atol=3e-2, rtol=2e-2)


@pytest.mark.parametrize("shape", [0, 1, 2, 3])
@pytest.mark.parametrize("beside", [0, 1, 6])
@pytest.mark.parametrize("m, n, k", [(65, 509, 96), (130, 1018, 160), (257, 38, 64)])
def test_tiled_product_off_steps_of_four(m, n, k, beside, shape):
    """Outputs and row strides off steps of 4: every result in its place, nothing written beside them.  A sum of k exact products
    is within k roundings of its terms, a stored bfloat16 half a unit in its last place further."""
    from qwen25vl_lite_amd.ops import tile
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, device="cuda", generator=g).bfloat16()
    w = (torch.randn(n, k, device="cuda", generator=g) / k ** 0.5).bfloat16()
    want = x.double() @ w.double().T
    bound = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    for dtype, last in ((torch.float32, 0.0), (torch.bfloat16, 2.0 ** -8)):
        room = torch.full((m + 2, 8 + n + beside), 7.0, device="cuda", dtype=dtype)
        inside = room.view(-1)[8:][:m * (8 + n + beside)].view(m, 8 + n + beside)[:, :n]
        tile.tile_product(x, w, dtype, out=inside, shape=shape)
        assert bool(((inside.double() - want).abs() <= bound + last * want.abs()).all())
        inside.fill_(7.0)
        assert bool((room == 7.0).all())
    if n % 2:
        return
    g, u = want[:, :n // 2].clamp(max=1.5), want[:, n // 2:].clamp(-1.5, 1.5)
    ref = g * torch.sigmoid(1.25 * g) * (u + 1.0)
    slack = 1.13 * 2.5 * bound[:, :n // 2] + 1.5 * bound[:, n // 2:]      # (slopes: see the rows kernel's test)
    got = tile.tile_gated(x, w, 1.25, 1.5, 1.0, shape=shape).double()
    assert bool(((got - ref).abs() <= slack + (2.0 ** -8 + 1e-6) * ref.abs() + 2e-6).all())


@pytest.mark.parametrize("shape, bn, bm", [(4, 192, 192), (5, 128, 192), (6, 192, 256), (7, 192, 320), (8, 128, 320), (9, 256, 192)])
@pytest.mark.parametrize("rows, outputs, k", [(-1, -2, 32), (1, 16, 64), (-80, 2, 96), (-126, -94, 160), (64, 48, 192)])
def test_tiled_product_in_shapes_that_do_not_halve(shape, bn, bm, rows, outputs, k):
    """Shapes whose halves are unequal or whose rows no number of whole fetches brings: rows and outputs around a tile's edges, an
    odd and an even number of steps, a last one of half its size.  A sum of k exact products is within k roundings of its terms."""
    from qwen25vl_lite_amd.ops import tile
    m, n = bm + rows, bn + outputs
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, device="cuda", generator=g).bfloat16()
    w = (torch.randn(n, k, device="cuda", generator=g) / k ** 0.5).bfloat16()
    want = x.double() @ w.double().T
    bound = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    for dtype, last in ((torch.float32, 0.0), (torch.bfloat16, 2.0 ** -8)):
        got = tile.tile_product(x, w, dtype, shape=shape).double()
        assert bool(((got - want).abs() <= bound + last * want.abs()).all())
    slope = 1.13 * (1.0 + 2.0 ** -8)
    if n % 16 == 0:
        two, b = want.view(m, n // 16, 2, 8), bound.view(m, n // 16, 2, 8)
        ref = torch.nn.functional.silu(two[:, :, 0]) * two[:, :, 1]
        slack = slope * (b[:, :, 0] * (two[:, :, 1].abs() + b[:, :, 1]) + two[:, :, 0].abs() * b[:, :, 1])
        got = tile.tile_swiglu(x, w, shape=shape).double().view(m, n // 16, 8)
        assert bool(((got - ref).abs() <= slack + (2.0 ** -8 + 1e-5) * ref.abs() + 2e-6).all())
    g, u = want[:, :n // 2].clamp(max=1.5), want[:, n // 2:].clamp(-1.5, 1.5)
    ref = g * torch.sigmoid(1.25 * g) * (u + 1.0)
    slack = 1.13 * 2.5 * bound[:, :n // 2] + 1.5 * bound[:, n // 2:]
    got = tile.tile_gated(x, w, 1.25, 1.5, 1.0, shape=shape).double()
    assert bool(((got - ref).abs() <= slack + (2.0 ** -8 + 1e-6) * ref.abs() + 2e-6).all())


@pytest.mark.parametrize("shape, bn, bm", [(0, 256, 256), (1, 128, 256), (2, 256, 128), (3, 128, 128), (4, 192, 192), (5, 128, 192), (6, 192, 256), (7, 192, 320),
                                           (8, 128, 320), (9, 256, 192)])
@pytest.mark.parametrize("k, splits", [(160, 3), (96, 2), (608, 9), (1056, 12), (1024, 7)])
def test_tiled_product_in_ranges_of_every_shape(shape, bn, bm, k, splits):
    """Ranges that do not divide the steps of 64, of one step and of several, with a last one of half its size: each slab holds its
    own range's sums, a sum of k exact products within k roundings of its terms."""
    from qwen25vl_lite_amd.ops import tile
    m, n = bm + 33, bn + 22
    g = torch.Generator(device="cuda").manual_seed(shape + k)
    x = torch.randn(m, k, device="cuda", generator=g).bfloat16()
    w = (torch.randn(n, k, device="cuda", generator=g) / k ** 0.5).bfloat16()
    out = torch.full((splits, m, n), math.nan, device="cuda")
    tile._launch(x, w, out, n, tile._SLABS, splits=splits, shape=shape)
    steps = (k + 63) // 64
    for i in range(splits):
        at = slice(64 * (steps * i // splits), 64 * (steps * (i + 1) // splits))
        a, b = x[:, at].double(), w[:, at].double()
        assert bool(((out[i].double() - a @ b.T).abs() <= k * 2.0 ** -24 * (a.abs() @ b.abs().T)).all()), i


@pytest.mark.parametrize("m", [1, 19, 40])
@pytest.mark.parametrize("n", [2, 34, 16401, 40970])
def test_rows_with_a_last_output_alone(m, n):
    """An odd number of outputs, or of channels of a gated product: the last one has no neighbour to be stored with."""
    from qwen25vl_lite_amd.ops import rows
    torch.manual_seed(m + n)
    k = 72
    x = torch.randn(m, k, device="cuda").bfloat16()
    w = (torch.randn(n, k, device="cuda") / math.sqrt(k)).bfloat16()
    want = x.double() @ w.double().T
    bound = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    for wider in (n % 2, 1 - n % 2):       # an even row stride, whose results are stored in pairs, and an odd one
        room = torch.full((m + 1, n + wider), 7.0, device="cuda").bfloat16()
        rows.rows_product(x, w, out=room[:m, :n])
        assert bool(((room[:m, :n].double() - want).abs() <= bound + 2.0 ** -8 * want.abs()).all())
        assert bool((room[:m, n:] == 7.0).all()) and bool((room[m] == 7.0).all())
    if n % 2:
        return
    got = rows.rows_gated(x, w, 1.25, 1.5, 1.0).double()
    g, u = want[:, :n // 2].clamp(max=1.5), want[:, n // 2:].clamp(-1.5, 1.5)
    ref = g * torch.sigmoid(1.25 * g) * (u + 1.0)
    slack = 1.13 * 2.5 * bound[:, :n // 2] + 1.5 * bound[:, n // 2:]
    assert bool(((got - ref).abs() <= slack + (2.0 ** -8 + 1e-6) * ref.abs() + 2e-6).all())


@pytest.mark.parametrize("m, n, k", [(65, 3584, 18944), (280, 2048, 11008), (100, 2560, 2048), (700, 272, 1376)])
def test_tiled_product_in_ranges(m, n, k):
    """Sums over ranges of the inner size that do not divide evenly, in float32 slabs; through the entry that joins them to
    the residual sum too."""
    from qwen25vl_lite_amd.ops import kernels, tile
    from qwen25vl_lite_amd.ops.linear import linear_into
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, device="cuda", generator=g).bfloat16()
    w = (torch.randn(n, k, device="cuda", generator=g) * 2 / k ** 0.5).bfloat16()
    want = x.float() @ w.float().T
    slabs = tile.tile_slabs(x, w)
    assert slabs is not None and slabs.shape[0] > 1 and slabs.dtype == torch.float32
    assert torch.allclose(slabs.sum(0), want, atol=3e-5, rtol=1e-4)
    h = torch.randn(m, n, device="cuda", generator=g)
    gain = torch.rand(n, device="cuda", generator=g) + 0.5
    total = h + want
    normed = kernels.add_rmsnorm(h, linear_into(h, x, w), gain, 1e-6, torch.float32)
    assert torch.allclose(h, total, atol=3e-5, rtol=1e-4)
    ref = total * torch.rsqrt(total.pow(2).mean(-1, keepdim=True) + 1e-6) * gain
    assert torch.allclose(normed, ref, atol=1e-4, rtol=1e-4)


@pytest.mark.parametrize("m, n, k", [(20, 50, 512), (33, 51, 1032), (64, 1, 2056), (100, 50, 512), (100, 49, 1024), (300, 37, 2080)])
def test_products_of_any_width_join_the_residual_sum(m, n, k):
    """Widths off steps of 4: what linear_into hands on, as slabs too, is taken by the norm behind it, whole and for chosen
    rows.  Each sum of k products and the addition into the residual is within k + 1 roundings of its terms."""
    from qwen25vl_lite_amd.ops import kernels
    from qwen25vl_lite_amd.ops.linear import linear_into
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, device="cuda", generator=g).bfloat16()
    w = (torch.randn(n, k, device="cuda", generator=g) / k ** 0.5).bfloat16()
    h = torch.randn(m, n, device="cuda", generator=g)
    gain = torch.rand(n, device="cuda", generator=g) + 0.5
    total = h.double() + x.double() @ w.double().T
    slack = (k + 1) * 2.0 ** -24 * (h.double().abs() + x.double().abs() @ w.double().abs().T)
    left = linear_into(None, x, w)
    if left.dtype == torch.bfloat16:              # uncut: one rounding of the product
        slack = slack + 2.0 ** -8 * (total - h.double()).abs()
    ref = total * torch.rsqrt(total.pow(2).mean(-1, keepdim=True) + 1e-6) * gain
    rows = torch.tensor([m - 1, 0], dtype=torch.int32, device="cuda")
    picked = kernels.add_rmsnorm(h, left, gain, 1e-6, torch.float32, rows=rows)
    normed = kernels.add_rmsnorm(h, left, gain, 1e-6, torch.float32)
    assert bool(((h.double() - total).abs() <= slack).all())
    # (a row's scale follows its sums: no term of it is off by more than the largest relative error of a row of one value)
    assert torch.allclose(normed.double(), ref, atol=2e-2 if left.dtype == torch.bfloat16 else 1e-3, rtol=1e-2)
    assert torch.equal(picked, normed[rows.long()])


def test_tiled_product_leaves_what_it_does_not_take():
    """Inner sizes off a step of 32, rows off 16 bytes, few rows: not taken, and the general entry still answers."""
    from qwen25vl_lite_amd.ops import tile
    from qwen25vl_lite_amd.ops.linear import linear
    torch.manual_seed(0)
    for m, n, k, off in ((100, 8192, 40, 0), (100, 8192, 64, 4), (64, 65536, 64, 0)):
        x = torch.randn(m, k + off, device="cuda").bfloat16()[:, off:]
        w = torch.randn(n, k, device="cuda").bfloat16()
        assert not tile.prefers_tile(x, w)
        assert torch.allclose(linear(x, w, out_dtype=torch.float32), x.float() @ w.float().T, atol=1e-3, rtol=1e-3)
