"""Rows that a product leaves for the norm behind it: which layers hand them on and which do not, with parts that compute on the CPU.

The parts defined here keep to the interfaces of ``parts/base.py``: a product that adds into the residual leaves ``h * gain`` and one over the
rows' root mean squares for the norm in ``step.ahead``, and a product takes such rows or normed ones.  Whatever hands on or not, a pass gives the same.
"""

from types import SimpleNamespace

import pytest
import torch

from qwen25vl_lite_amd.models import DecoderModel, LayerSpec, ModelSpec, RunEntry
from qwen25vl_lite_amd.parts import (Block, Embedding, FeedForward, Head, Mixer, Norm, ParamSpec, PartSpec, build_part, known_parts, register_part)
from qwen25vl_lite_amd.parts.block import PreNormBlock

HIDDEN, VOCAB = 12, 20
calls = []                       # what ran, in order: "norm <name>" and "taken <name>" (rows that were left, in place of a norm)


class Left:
    def __init__(self, rows, by):
        self.rows, self.by = rows, by


class ToyNorm(Norm):
    def __init__(self, params, dtype, device):
        super().__init__(dtype, device)
        self.name = params["name"]

    def param_specs(self):
        return {"weight": ParamSpec((HIDDEN,), "vector")}

    def load(self, tensors):
        self.weight = tensors["weight"]

    def forward(self, stream, rows=None, lazy=False):
        for term in (stream.pending, stream.row_addend):
            if term is not None:
                stream.h += term
        stream.pending = stream.row_addend = None
        calls.append("norm " + self.name)
        h = stream.h if rows is None else stream.h[rows.long()]
        return h * self.weight * torch.rsqrt(h.pow(2).mean(1, keepdim=True) + 1e-6)

    def ahead(self):
        return SimpleNamespace(weight=self.weight, name=self.name, left=None)


class ToyProduct:
    leaves_ahead = True
    bias = False                 # with one the product is handed back, as an output projection with a bias is

    def __init__(self, params, dtype, device):
        super().__init__(dtype, device)

    def param_specs(self):
        return {"weight": ParamSpec((HIDDEN, HIDDEN))}

    def load(self, tensors):
        self.weight = tensors["weight"]

    def takes_scaled(self, rows):
        return rows <= 16

    def forward(self, x, step, slot=None):
        y = torch.tanh(x.rows @ self.weight * x.by if isinstance(x, Left) else x @ self.weight)
        if step.residual is None or self.bias:
            return y
        step.residual += y
        if step.ahead is not None:
            h = step.residual
            step.ahead.left = Left(h * step.ahead.weight, torch.rsqrt(h.pow(2).mean(1, keepdim=True) + 1e-6))
            calls.append("taken " + step.ahead.name)
        return None


class ToyMixer(ToyProduct, Mixer):
    pass


class ToyFeedForward(ToyProduct, FeedForward):
    pass


class ToyEmbedding(Embedding):
    def __init__(self, params, dtype, device):
        super().__init__(dtype, device)

    def param_specs(self):
        return {"weight": ParamSpec((VOCAB, HIDDEN), "table")}

    def load(self, tensors):
        self.table = tensors["weight"]

    def forward(self, token_ids, step):
        return self.table[token_ids.long()].clone()


class ToyHead(Head):
    def __init__(self, params, dtype, device):
        super().__init__(dtype, device)

    def param_specs(self):
        return {"weight": ParamSpec((VOCAB, HIDDEN))}

    def load(self, tensors):
        self.weight = tensors["weight"]

    def forward(self, x, step):
        return x @ self.weight.T


class OtherNorm(ToyNorm):
    """A norm with a forward of its own that says nothing about rows left for it."""

    def forward(self, stream, rows=None, lazy=False):
        return 0.5 * super().forward(stream, rows, lazy) + 0.25


class OtherMixer(ToyMixer):
    """Adds something else behind the product, to a sum that it may change in place."""

    def forward(self, x, step, slot=None):
        y = super().forward(x, step, slot)
        step.residual += 0.125
        return y


class OtherFeedForward(ToyFeedForward):
    """Reads normed rows as a tensor."""

    def forward(self, x, step, slot=None):
        return super().forward(x * 1.5, step, slot)


class BiasedMixer(ToyMixer):
    bias = True


class OtherBlock(PreNormBlock):
    """An arrangement of its own, by what a block was asked for before rows could be left."""

    def forward(self, stream, step, slot):
        x = self.norm1.forward(stream)
        step.residual = None
        stream.pending = self.mixer.forward(x, step, slot)
        y = self.norm2.forward(stream)
        stream.pending = self.ffn.forward(y, step)
        return stream


class Twice(Block):
    """Two layers in one."""

    def __init__(self, params, dtype, device):
        super().__init__(dtype, device)
        self.a, self.b = (build_part("block", params[k], dtype, device) for k in ("a", "b"))

    def sub_parts(self):
        return {"a": self.a, "b": self.b}

    def forward(self, stream, step, slot):
        return self.b.forward(self.a.forward(stream, step, slot), step, slot)


for _category, _kind, _part in (("norm", "cpu_norm", ToyNorm), ("norm", "cpu_norm_other", OtherNorm), ("mixer", "cpu_mixer", ToyMixer),
                                ("mixer", "cpu_mixer_other", OtherMixer), ("mixer", "cpu_mixer_biased", BiasedMixer), ("ffn", "cpu_ffn", ToyFeedForward),
                                ("ffn", "cpu_ffn_other", OtherFeedForward), ("embedding", "cpu_embedding", ToyEmbedding), ("head", "cpu_head", ToyHead),
                                ("block", "cpu_block_other", OtherBlock), ("block", "cpu_twice", Twice)):
    if _kind not in known_parts(_category):
        register_part(_category, _kind, _part)


def _layer(name, norm1="cpu_norm", mixer="cpu_mixer", norm2="cpu_norm", ffn="cpu_ffn", block="pre_norm"):
    return PartSpec(block, {"norm1": PartSpec(norm1, {"name": name + "1"}), "mixer": PartSpec(mixer, {}), "norm2": PartSpec(norm2, {"name": name + "2"}),
                            "ffn": PartSpec(ffn, {}), "names": {"norm1": "n1", "mixer": "m", "norm2": "n2", "ffn": "f"}})


def _run(layers, run=None, rows=3, **more):
    """``(logits, what ran)`` as it is and with nothing handed on."""
    spec = ModelSpec(hidden_size=HIDDEN, vocab_size=VOCAB, layers=[LayerSpec(s, f"l{i}.") for i, s in enumerate(layers)],
                     run=run or [RunEntry(i) for i in range(len(layers))], final_norm=PartSpec("cpu_norm", {"name": "end"}), tie_word_embeddings=False,
                     embed=PartSpec("cpu_embedding", {}), head=PartSpec("cpu_head", {}), **more)
    model = DecoderModel(spec, torch.float32, "cpu")
    g = torch.Generator().manual_seed(3)
    for part, names in model.part_groups():
        model.load_part(part, {k: torch.randn(model.expected_tensors()[n].shape, generator=g) for k, n in names.items()})
    from qwen25vl_lite_amd.parts import LayerSlot, StepContext
    none = torch.zeros(0, dtype=torch.int32)
    results = []
    for takes in (ToyProduct.takes_scaled, lambda self, rows: False):
        with pytest.MonkeyPatch.context() as patch:
            patch.setattr(ToyProduct, "takes_scaled", takes)
            step = StepContext(num_tokens=rows, num_reqs=rows, token_ids=torch.arange(rows, dtype=torch.int32) % VOCAB, positions=none, token_req=none,
                               token_seqpos=none, cu_q=none, ctx_len=none, req_slots=none, groups=[], logit_rows=torch.arange(rows, dtype=torch.int32))
            del calls[:]
            logits = model.forward(step, [LayerSlot() for _ in model.spec.run])
            results.append((logits, list(calls)))
    (got, ran), (want, plain) = results
    assert not any(c.startswith("taken") for c in plain)
    assert torch.allclose(got, want, rtol=1e-4, atol=1e-4), (ran, (got - want).abs().max())     # (the same sums, a row divided before or behind them)
    return ran


def test_every_norm_between_two_products():
    ran = _run([_layer("a"), _layer("b"), _layer("c")])
    assert ran == ["norm a1", "taken a2", "taken b1", "taken b2", "taken c1", "taken c2", "norm end"]


def test_a_layer_that_runs_again():
    ran = _run([_layer("a"), _layer("b")], run=[RunEntry(0), RunEntry(1), RunEntry(0), RunEntry(0)])
    assert ran == ["norm a1", "taken a2", "taken b1", "taken b2", "taken a1", "taken a2", "taken a1", "taken a2", "norm end"]


def test_more_rows_than_the_products_take():
    assert not any(c.startswith("taken") for c in _run([_layer("a"), _layer("b")], rows=17))


def test_a_sum_that_changes_before_the_next_layer():
    """A vector added to every row, the embedding's output mixed in: the next layer's first norm reads the changed sum."""
    run = [RunEntry(0), RunEntry(1, add_vector=1), RunEntry(0)]
    ran = _run([_layer("a"), _layer("b")], run=run, pass_vectors_name="vectors.weight", pass_vectors_rows=2)
    assert ran == ["norm a1", "taken a2", "norm b1", "taken b2", "taken a1", "taken a2", "norm end"]


def test_the_embedding_mixed_in(monkeypatch):
    from qwen25vl_lite_amd.models import decoder
    from qwen25vl_lite_amd.parts import ResidualStream
    monkeypatch.setattr(decoder.PassMix, "from_first", lambda self, x0: x0 @ self.w_first.T)

    def mixed(self, stream, share):
        h = stream.h if stream.pending is None else stream.h + stream.pending
        return ResidualStream(h @ self.w_sum.T, pending=share)
    monkeypatch.setattr(decoder.PassMix, "forward", mixed)
    ran = _run([_layer("a"), _layer("b")], run=[RunEntry(0), RunEntry(1, mix_input=True), RunEntry(0)], pass_mix_name="mix.weight")
    assert ran == ["norm a1", "taken a2", "norm b1", "taken b2", "taken a1", "taken a2", "norm end"]


def test_a_product_that_is_handed_back():
    """An output projection with a bias does not add in place and leaves nothing: the norm behind it runs."""
    assert _run([_layer("a", mixer="cpu_mixer_biased"), _layer("b")]) == ["norm a1", "norm a2", "taken b1", "taken b2", "norm end"]


@pytest.mark.parametrize("what, ran", [
    (dict(norm1="cpu_norm_other"), ["norm a1", "taken a2", "norm b1", "taken b2", "taken c1", "taken c2", "norm end"]),
    (dict(norm2="cpu_norm_other"), ["norm a1", "taken a2", "taken b1", "norm b2", "taken c1", "taken c2", "norm end"]),
    (dict(mixer="cpu_mixer_other"), ["norm a1", "taken a2", "norm b1", "norm b2", "taken c1", "taken c2", "norm end"]),
    (dict(ffn="cpu_ffn_other"), ["norm a1", "taken a2", "taken b1", "norm b2", "norm c1", "taken c2", "norm end"]),
    (dict(block="cpu_block_other"), ["norm a1", "taken a2", "norm b1", "norm b2", "norm c1", "taken c2", "norm end"])])
def test_a_subclass_with_a_forward_of_its_own(what, ran):
    """What a class says about its forward does not hold for a subclass's."""
    assert _run([_layer("a"), _layer("b", **what), _layer("c")]) == ran


def test_layers_within_a_layer():
    """The rows that the next layer's norm asks for are left by the layer in front of it, not by one inside that: what a layer within hands on, nobody
    asked for."""
    twice = PartSpec("cpu_twice", {"a": _layer("b"), "b": _layer("c")})
    assert _run([_layer("a"), twice, _layer("d")]) == ["norm a1", "taken a2", "norm b1", "taken b2", "norm c1", "taken c2", "norm d1", "taken d2", "norm end"]
