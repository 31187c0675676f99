"""Decoded tokens whose tile eight waves share (csrc/attention_window.hip): against four waves, and against 64 bits where nothing but a causal mask is asked for."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# contexts of one key, fewer blocks of 32 than waves, as many, one key more, many; sizes of keys and values with one, several and a part of a tile of channels
@pytest.mark.parametrize("hd, vd, nq, nkv", [(128, 128, 28, 4), (16, 24, 6, 2), (256, 192, 28, 1), (64, 32, 16, 16)])
@pytest.mark.parametrize("window, keep, chunk, sunk, turned", [(None, 0, None, False, False), (300, 5, None, True, False), (None, 0, 290, False, True)])
def test_eight_waves_a_tile(hd, vd, nq, nkv, window, keep, chunk, sunk, turned):
    from qwen25vl_lite_amd.ops import attention_window
    from qwen25vl_lite_amd.parts import StepContext
    lens, ps = [1, 33, 224, 256, 257, 300, 513, 900], 16
    b, need, g = len(lens), [(n + 15) // 16 for n in lens], torch.Generator().manual_seed(hd + vd)
    k, v = (torch.randn(sum(need) * ps, nkv, width, generator=g).bfloat16() for width in (hd, vd))
    q = torch.randn(b, nq, hd, generator=g).bfloat16()
    table, at, want = torch.full((b, max(need)), -1, dtype=torch.int32), 0, []
    for i, n in enumerate(lens):
        table[i, :need[i]] = torch.arange(at, at + need[i])
        kk, vv = (t[at * ps:at * ps + n].double().repeat_interleave(nq // nkv, 1) for t in (k, v))
        p = torch.softmax((kk * q[i].double()).sum(2) * hd ** -0.5, 0)
        want.append((p[:, :, None] * vv).sum(0).reshape(-1))
        at += need[i]
    kc = k.view(-1, ps, nkv, hd).permute(0, 2, 1, 3).contiguous().cuda()
    vc = v.view(-1, ps, nkv, vd).permute(0, 2, 3, 1).contiguous().cuda()
    cu, none = list(range(b + 1)), torch.zeros(0, dtype=torch.int32).cuda()
    step = StepContext(num_tokens=b, num_reqs=b, token_ids=none, positions=none, token_req=none, token_seqpos=none,
                       cu_q=torch.tensor(cu, dtype=torch.int32).cuda(), ctx_len=torch.tensor(lens, dtype=torch.int32).cuda(), req_slots=none, groups=[],
                       logit_rows=none, cu_q_host=cu, ctx_len_host=lens, max_q_len=1, max_ctx_len=max(lens), dtype=torch.bfloat16)
    angles = torch.rand(b, vd // 2, generator=g) * 6
    extra = dict(sinks=torch.linspace(-1, 2, nq).cuda() if sunk else None, chunk=chunk,
                 turn=torch.stack([angles.cos(), angles.sin()], 2).contiguous().cuda() if turned else None)
    four, eight, chosen = (attention_window.try_attention(q.view(b, -1).cuda(), kc, vc, table.cuda(), step, nq, window, keep, hd ** -0.5, share=s, **extra)
                           .double().cpu() for s in (1, 2, None))
    assert torch.equal(chosen, eight)          # more keys than EIGHT_WAVES_FROM in the longest walk, few tiles
    # probabilities are rounded to bfloat16 (a weighted mean of values below 5: half a unit in the last place of 5 at most), and the result
    slack = 5 * 2.0 ** -9 + 2.0 ** -10
    assert bool(((eight - four).abs() <= 2.0 ** -7 * four.abs() + 2 * slack).all())
    if window is None and chunk is None:
        assert bool(((eight - torch.stack(want)).abs() <= 2.0 ** -8 * torch.stack(want).abs() + slack).all())
