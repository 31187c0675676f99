"""More blocks than compute units with short walks, in blocks of half the waves (csrc/attention_mfma.hip): against blocks of all and the oracle."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _with_sinks(c, nq, nkv, window, sinks):
    """In 64 bits, token by token out of the pages: a head's sink joins the denominator and brings no value."""
    rows = []
    for i, (r, p) in enumerate(zip(c["req"].tolist(), c["seqpos"].tolist())):
        first, pages = 0 if window is None else max(0, p - window + 1), c["table"][r].long()
        pages = pages[:p // 16 + 1]
        k = c["kc"][pages].double().permute(1, 0, 2, 3).reshape(nkv, -1, 128)[:, first:p + 1].repeat_interleave(nq // nkv, 0)
        v = c["vc"][pages].double().permute(1, 0, 3, 2).reshape(nkv, -1, 128)[:, first:p + 1].repeat_interleave(nq // nkv, 0)
        scores = (k @ c["q"][i].double().view(nq, 128, 1)).squeeze(2) * c["scale"]
        weights = torch.softmax(torch.cat([scores, sinks.double()[:, None]], 1), 1)[:, :-1]
        rows.append((weights[:, None] @ v).reshape(-1))
    return torch.stack(rows).float().cpu()


# one key more than waves' blocks of 32 hold, contexts that end inside a block, prompts that end inside a tile, a last one of the longest that goes this way
@pytest.mark.parametrize("lens, qlens", [((129, 33, 1, 257), (129, 33, 1, 57)), ((512, 300, 31, 64), (1, 130, 31, 17)), ((96,) * 4, (48,) * 4)])
@pytest.mark.parametrize("nq, nkv, window, sunk", [(16, 2, None, False), (14, 2, 100, False), (8, 8, None, True), (4, 1, 7, True)])
def test_half_the_waves(lens, qlens, nq, nkv, window, sunk, monkeypatch):
    from qwen25vl_lite_amd.ops import attention_mfma
    from qwen25vl_lite_amd.parts import StepContext
    from test_gpu_kernels import _attention_case
    c = _attention_case(torch.bfloat16, nq, nkv, 128, window, lens, qlens)
    monkeypatch.setattr(attention_mfma, "plan_splits", lambda t, n, m, d=None: ("coop", 1, 0))
    cu = [0]
    for n in qlens:
        cu.append(cu[-1] + n)
    none = torch.zeros(0, dtype=torch.int32).cuda()
    sinks, outs = torch.linspace(-1, 2, nq).cuda() if sunk else None, []
    for fill in (0, 1 << 20):                  # more blocks than this: half the waves
        monkeypatch.setattr(attention_mfma, "FILL_BLOCKS", fill)
        before = attention_mfma.taken.copy()
        step = StepContext(num_tokens=cu[-1], num_reqs=4, token_ids=none, positions=none, token_req=c["req"], token_seqpos=c["seqpos"],
                           cu_q=torch.tensor(cu, dtype=torch.int32).cuda(), ctx_len=torch.tensor(lens, dtype=torch.int32).cuda(), req_slots=none, groups=[],
                           logit_rows=none, cu_q_host=cu, ctx_len_host=list(lens), max_q_len=max(qlens), max_ctx_len=max(lens), dtype=torch.bfloat16)
        outs.append(attention_mfma.try_attention(c["q"], c["kc"], c["vc"], c["table"], step, nq, window, c["scale"], sinks=sinks).float().cpu())
        assert attention_mfma.taken - before == {"shared tiles, half the waves" if fill == 0 else "shared tiles": 1}
    want = c["want"] if sinks is None else _with_sinks(c, nq, nkv, window, sinks)
    assert torch.allclose(outs[0], want, atol=1.5e-2, rtol=2e-2)
    # the same keys' probabilities in other waves: each is rounded to bfloat16 against another reference, as are the sums that are written
    assert torch.allclose(outs[0], outs[1], atol=1.5e-2, rtol=2e-2)
