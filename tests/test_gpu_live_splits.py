"""Decoded tokens whose blocks share the keys that are there (csrc/attention_mfma.hip): splits of a step that was planned for longer contexts."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


# contexts of one key, a block of 32 and one key beside it, of what one split holds, of one key more, of all splits; fewer splits than are merged at a time (two, four,
# eight), as many, more; splits that are empty, and the window's first key inside a block of 32
@pytest.mark.parametrize("nsplit, least", [(2, 32), (3, 64), (4, 128), (5, 32), (9, 32), (17, 64)])
@pytest.mark.parametrize("nq, nkv, hd, window", [(14, 2, 128, None), (6, 2, 48, 100), (8, 8, 16, 7), (4, 1, 192, None)])
@pytest.mark.parametrize("counted", [True, False])
def test_splits_of_the_keys_that_are_there(nsplit, least, nq, nkv, hd, window, counted, monkeypatch):
    from qwen25vl_lite_amd.ops import attention_mfma
    from qwen25vl_lite_amd.parts import StepContext
    lens, ps = [1, 31, 32, 33, 64, 65, 128, 129, 333, 640, 1025], 16
    b, width = len(lens), 1040 // ps
    g = torch.Generator().manual_seed(nsplit * hd)
    need = [(n + ps - 1) // ps for n in lens]
    k, v = (torch.randn(sum(need) * ps, nkv, hd, generator=g).bfloat16() for _ in range(2))
    q = torch.randn(b, nq, hd, generator=g).bfloat16()
    table, at, want = torch.full((b, width), -1, dtype=torch.int32), 0, []
    for i, n in enumerate(lens):
        table[i, :need[i]] = torch.arange(at, at + need[i])
        first = 0 if window is None else max(0, n - window)
        kk, vv = k[at * ps + first:at * ps + n].double(), v[at * ps + first:at * ps + n].double()
        kk, vv = kk.repeat_interleave(nq // nkv, 1), vv.repeat_interleave(nq // nkv, 1)
        p = torch.softmax((kk * q[i].double()).sum(2) * hd ** -0.5, 0)
        want.append((p[:, :, None] * vv).sum(0).reshape(-1))
        at += need[i]
    want = torch.stack(want)
    kc = k.view(-1, ps, nkv, hd).permute(0, 2, 1, 3).contiguous().cuda()
    vc = v.view(-1, ps, nkv, hd).permute(0, 2, 3, 1).contiguous().cuda()
    if not counted:
        monkeypatch.setattr(attention_mfma, "MERGE_COUNTERS", 0)
    monkeypatch.setattr(attention_mfma, "plan_splits", lambda t, n, m, d=None: ("coop", nsplit, least))
    cu, none = list(range(b + 1)), torch.zeros(0, dtype=torch.int32).cuda()
    step = StepContext(num_tokens=b, num_reqs=b, token_ids=none, positions=none, token_req=none, token_seqpos=none,
                       cu_q=torch.tensor(cu, dtype=torch.int32).cuda(), ctx_len=torch.tensor(lens, dtype=torch.int32).cuda(), req_slots=none, groups=[],
                       logit_rows=none, cu_q_host=cu, ctx_len_host=[2048] * b, max_q_len=1, max_ctx_len=2048, lengths_known=False, dtype=torch.bfloat16)
    rows = q.view(b, nq * hd).cuda()
    outs = [attention_mfma.try_attention(rows, kc, vc, table.cuda(), step, nq, window, hd ** -0.5) for _ in range(3)]
    # probabilities are rounded to bfloat16 (a weighted mean of values below 5: half a unit in the last place of 5 at most), and the result
    assert bool(((outs[0].double().cpu() - want).abs() <= 2.0 ** -8 * want.abs() + 5 * 2.0 ** -9 + 2.0 ** -10).all())
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])      # the counters are at zero each time
    if counted:
        assert int(attention_mfma._counters(rows.device).abs().sum()) == 0


@pytest.mark.parametrize("counted", [True, False])
@pytest.mark.parametrize("window", [None, 7])
def test_a_row_without_keys_is_written(counted, window, monkeypatch):
    """A request whose context is empty, between others: with sinks every probability goes there and its row is zeros, whatever the memory held."""
    from qwen25vl_lite_amd.ops import attention_mfma
    from qwen25vl_lite_amd.parts import StepContext
    lens, ps, nq, nkv, hd = [40, 0, 100], 16, 4, 2, 128
    if not counted:
        monkeypatch.setattr(attention_mfma, "MERGE_COUNTERS", 0)
    monkeypatch.setattr(attention_mfma, "plan_splits", lambda t, n, m, d=None: ("coop", 4, 32))
    g = torch.Generator(device="cuda").manual_seed(5)
    kc, vc, rows = (torch.randn(*s, device="cuda", generator=g).bfloat16() for s in ((8, nkv, ps, hd), (8, nkv, hd, ps), (3, nq * hd)))
    table = torch.arange(24, device="cuda", dtype=torch.int32).view(3, 8) % 8
    cu, none = [0, 1, 2, 3], torch.zeros(0, dtype=torch.int32).cuda()
    step = StepContext(num_tokens=3, num_reqs=3, token_ids=none, positions=none, token_req=none, token_seqpos=none,
                       cu_q=torch.tensor(cu, dtype=torch.int32).cuda(), ctx_len=torch.tensor(lens, dtype=torch.int32).cuda(), req_slots=none, groups=[],
                       logit_rows=none, cu_q_host=cu, ctx_len_host=[1024] * 3, max_q_len=1, max_ctx_len=1024, lengths_known=False, dtype=torch.bfloat16)
    made, sinks = [], torch.linspace(-1, 2, nq).cuda()

    def filled(like):
        made.append(torch.full_like(like, 7.0))
        return made[-1]
    monkeypatch.setattr(attention_mfma.torch, "empty_like", filled)
    out = attention_mfma.try_attention(rows, kc, vc, table, step, nq, window, hd ** -0.5, sinks=sinks)
    assert out is made[-1] and bool((out[1] == 0).all()) and bool((out[[0, 2]] != 7.0).any(1).all())
    if counted:
        assert int(attention_mfma._counters(rows.device).abs().sum()) == 0
