"""Rows that a product leaves for the norm behind it, from the sum to the product that takes them: the rules on both sides of the row counts and sizes at
which they change, and layers whose norms have no kernel against the same layers with all of them."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


# outputs for a part of the compute units and more than 64 for each; inner sizes for one pass of a block and beyond, and one that small tiles do not take
@pytest.mark.parametrize("n, k", [(272, 2048), (272, 4104), (2048, 2048), (16400, 2048), (2048, 2568)])
def test_sums_that_leave_rows(n, k):
    from qwen25vl_lite_amd.ops import linear as products
    from qwen25vl_lite_amd.ops import mid, skinny, stream
    gain, eps = torch.randn(n, device="cuda"), 1e-6
    few = n <= 64 * min(256, torch.cuda.get_device_properties(0).multi_processor_count)
    for m in (1, 8, 9, 16, 17, 64, 65, 255, 256, 300):
        g = torch.Generator(device="cuda").manual_seed(m + n + k)
        x = torch.randn(m, k, device="cuda", generator=g).bfloat16()
        w = (torch.randn(n, k, device="cuda", generator=g) / math.sqrt(k)).bfloat16()
        want, slack = x.double() @ w.double().T, k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)      # k roundings of a sum's terms
        for asked in (True, False):
            for in_place in (True, False):
                h = torch.randn(m, n, device="cuda", generator=g)
                before, ahead = h.double(), products.NormAhead(gain, eps, torch.bfloat16) if asked else None
                left = products.linear_into(h, x, w, ahead, in_place=in_place)
                here, case = left is None, (m, asked, in_place)
                got = h.double() if here else before + (left.double().sum(0) if left.dim() == 3 else left.double())
                last = 2.0 ** -8 if not here and left.dtype == torch.bfloat16 else 2.0 ** -23
                assert bool(((got - (before + want)).abs() <= slack + last * (want.abs() + (before + want).abs())).all()), case
                if not here:
                    assert torch.equal(h.double(), before), case
                leaves = asked and ((m <= stream.MOST_ROWS and few) or (in_place and m > 64 and mid.prefers_into(m, k, w)))
                assert (ahead is not None and ahead.left is not None) == leaves, case
                if m <= stream.MOST_ROWS and few:
                    assert here == (asked or not skinny.prefers_split(m, k, w) or (in_place and m <= products.IN_PLACE_ROWS)), case
                if leaves:
                    rows = ahead.left
                    assert here and rows.h is h and torch.equal(rows.rows, (h * gain).bfloat16()), case
                    squares, parts, e = rows.scaled
                    exact = (h.double() ** 2).sum(1)
                    # sums of n squares, none negative: as many roundings at most
                    assert e == eps and bool(((squares[:, :parts].double().sum(1) - exact).abs() <= n * 2.0 ** -24 * exact).all()), case


@pytest.mark.parametrize("rows", [1, 8, 16, 17, 64, 300])
def test_layers_without_norm_kernels(rows, monkeypatch):
    """Three layers of width 2,048 over a prompt: which products take rows that were left, and the logits beside those of the same layers with every norm formed.

    What differs is where a row is divided by its root mean square.  In either, some 6 tensors of a layer are rounded to bfloat16 on the way, and a value that
    is rounded the other way moves by 2^-8 of itself."""
    from qwen25vl_lite_amd import EngineConfig, ModelRunner, build_model
    from qwen25vl_lite_amd.config import load_config
    from qwen25vl_lite_amd.engine.batch import StepEntry
    from qwen25vl_lite_amd.models import decoder
    from qwen25vl_lite_amd.ops import linear as products
    from qwen25vl_lite_amd.ops import skinny
    from qwen25vl_lite_amd.parts import block
    layers = 3
    model = build_model(load_config({
        "architectures": ["Qwen2_5_VLForConditionalGeneration"], "hidden_size": 2048, "intermediate_size": 6144, "num_hidden_layers": layers,
        "num_attention_heads": 16, "num_key_value_heads": 2, "vocab_size": 512, "tie_word_embeddings": False, "rms_norm_eps": 1e-6, "rope_theta": 1e6,
        "rope_scaling": {"type": "mrope", "mrope_section": [16, 24, 24]}}), torch.bfloat16, "cuda:0")
    g = torch.Generator(device="cuda").manual_seed(11)
    expected = model.expected_tensors()
    for part, names in model.part_groups():
        tensors = {}
        for local, name in names.items():
            shape = expected[name].shape
            t = torch.randn(shape, device="cuda", generator=g)
            if name.endswith("norm.weight"):
                tensors[local] = 0.5 + t.abs()
            else:
                tensors[local] = t if len(shape) == 1 else (t * (5.0 if name.startswith("embed") else 1.0 / math.sqrt(shape[1]))).bfloat16()
        model.load_part(part, tensors)
    taken = {}

    def counted(module, name, of):
        kept = getattr(module, name)

        def call(*args, **kw):
            scaled = kw.get("scaled", args[of] if len(args) > of else None)
            taken[name] = taken.get(name, 0) + (scaled is not None)
            return kept(*args, **kw)
        monkeypatch.setattr(module, name, call)
    counted(skinny, "slice_qkv_rope", 11)
    counted(products.stream, "stream_gated", 3)
    counted(products.tile, "tile_swiglu", 5)
    tokens = torch.randint(0, 512, (rows,), generator=torch.Generator().manual_seed(rows)).tolist()
    logits = []
    for hands_on in (True, False):
        if not hands_on:
            for module in (block, decoder):
                monkeypatch.setattr(module, "says", lambda part, name: False)
        runner = ModelRunner(model, EngineConfig(num_blocks=24, block_size=16, max_num_seqs=2, max_num_batched_tokens=512, max_model_len=384,
                                                 enable_prefix_cache=False, dtype=torch.bfloat16, device="cuda:0"))
        taken.clear()
        runner.admit(0)
        logits.append(runner.execute([StepEntry(0, tokens, 0, want=list(range(rows)))]).double())
        counts = tuple(taken.get(name, 0) for name in ("slice_qkv_rope", "stream_gated", "tile_swiglu"))
        few, many = hands_on and rows <= 16, hands_on and rows == 300
        assert counts == ((layers - 1) * few, layers * few, layers * many)
    a, b = logits
    assert float((a - b).norm() / b.norm()) <= layers * 6 * 2.0 ** -8
    if rows in (17, 64):
        assert torch.equal(a, b)
