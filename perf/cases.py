"""What a user of the engine has it do, as cases that can be timed and checked.

A case is one pass through the public entry points: ``ModelRunner`` steps over requests that share a
batch (``kind`` ``"steps"``), or the device sampler on a step's logits (``kind`` ``"sample"``).

A pass of steps works on two sorts of requests.  ``batch`` running requests stand at contexts of up to
``context`` tokens whose keys and values are in the cache (whole pages, as the prefix cache keeps them);
the pass forks each, so that it can be taken again from the same place.  ``arrivals`` new requests bring
prompts of up to ``prompt`` tokens, which are run in portions of at most ``budget`` tokens a step, beside
one token of every running request; a prompt that is through decodes from the next step on.  The pass ends
when all prompts are through and ``decode`` decode steps have been taken.  The tokens that are decoded are
given (the scoring of known continuations), so that a result is a matter of rounding and never of which of
two near equal logits was larger.  The logits of every decoded token and of every prompt's last are
the outputs.

Weights are random, at the layer sizes of the decoders that ``bench.py`` measures, with fewer of the equal
layers: what a layer costs does not depend on how many there are.
"""

from __future__ import annotations

import math
import zlib

import numpy as np
import torch

# Layer sizes of the Qwen2.5-VL 3B, 7B and 72B text decoders: width, feed-forward, query heads, key heads,
# vocabulary, tied head.  Heads have 128 channels.
SIZES = {"3b": (2048, 11008, 16, 2, 151936, True),
         "7b": (3584, 18944, 28, 4, 152064, False),
         "72b": (8192, 29568, 64, 8, 152064, False)}
HEAD = 128
PAGE = 16


# ------------------------------------------------------------------------------------------------ the cases
def steps_case(name=None, design="qwen25vl", size="7b", layers=8, dtype="bfloat16", batch=0, context=0, arrivals=0,
               prompt=0, budget=4096, decode=0):
    case = {"kind": "steps", "design": design, "size": size, "layers": layers, "dtype": dtype, "batch": batch,
            "context": context, "arrivals": arrivals, "prompt": prompt, "budget": budget, "decode": decode}
    return case if name is None else {"name": name, **case}


def sample_case(name=None, rows=64, vocab=152064):
    case = {"kind": "sample", "rows": rows, "vocab": vocab}
    return case if name is None else {"name": name, **case}


def listed():
    return [
        # every decoded token ends here: a batch whose requests ask for different things (greedy, top-p, top-k with
        # penalties, min-p)
        sample_case("sample_64", 64, 152064),
        # one user, a short question: the smallest step, where launches and latency count
        steps_case("decode_1_3b", size="3b", batch=1, context=32, decode=8),
        # the benchmark's own step: eight requests with 512-token prompts
        steps_case("decode_8_7b", batch=8, context=512, decode=16),
        # an odd number of requests on wide layers: rows for two tiles of the matrix instruction, long inner sizes
        steps_case("decode_19_72b", size="72b", layers=2, batch=19, context=1024, decode=4),
        # a full server: 64 requests at contexts of all lengths
        steps_case("decode_64_7b", batch=64, context=768, decode=8),
        # short questions that arrive together: a small ragged prefill, then nothing else
        steps_case("prompts_short_3b", size="3b", arrivals=5, prompt=120),
        # the benchmark's prefill
        steps_case("prompt_2048_7b", arrivals=1, prompt=2048),
        # a long document read in portions, and the first tokens of the answer
        steps_case("long_prompt_7b", layers=4, arrivals=1, prompt=12288, decode=6),
        # continuous batching: new prompts run in small portions beside requests that decode
        steps_case("mixed_3b", size="3b", batch=24, context=768, arrivals=4, prompt=300, budget=256, decode=6),
        # the exact mode: float32 weights and arithmetic throughout
        steps_case("float32_3b", size="3b", layers=2, dtype="float32", batch=4, context=64, arrivals=2, prompt=100,
                   budget=160, decode=4),
        # linear attention with per-head and per-channel decays: prompts, then decoding, one conversation turn
        steps_case("gogudra_7b", design="gogudra", layers=4, arrivals=8, prompt=300, decode=12),
        # routed experts, a latent cache, windows with sinks behind short convolutions
        steps_case("rofapel_7b", design="rofapel", layers=4, arrivals=8, prompt=384, decode=8),
    ]


def draw(rng):
    """A case of the same ranges: 1 to 64 requests, contexts of 16 to 2,048 tokens, prompts of 1 to 12,288, portions of 64
    to 4,096, any of the designs and sizes."""
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    most = max(_cost(c) for c in listed())
    while True:
        what = rng.choice(["sample", "decode", "decode", "prompts", "prompts", "mixed", "design", "design", "float32"])
        size = rng.choice(["3b", "7b", "7b"])
        if what == "sample":
            return sample_case(rows=spread(1, 64), vocab=SIZES[size][4])
        if what == "decode":
            size = rng.choice(["3b", "7b", "72b"])
            case = steps_case(size=size, layers=2 if size == "72b" else 8, batch=spread(1, 64), context=spread(16, 2048),
                              decode=rng.randint(3, 12))
        elif what == "prompts":
            case = steps_case(size=size, layers=4, arrivals=spread(1, 8), prompt=spread(1, 12288),
                              budget=rng.choice([1024, 2048, 4096]), decode=rng.choice([0, 0, 4]))
        elif what == "mixed":
            case = steps_case(size=size, layers=4, batch=spread(1, 48), context=spread(16, 2048), arrivals=spread(1, 6),
                              prompt=spread(8, 1024), budget=spread(64, 1024), decode=rng.randint(2, 6))
        elif what == "design":
            case = steps_case(design=rng.choice(["gogudra", "rofapel"]), size=size, layers=4, arrivals=spread(1, 16),
                              prompt=spread(1, 2048), decode=rng.randint(0, 10))
        else:
            case = steps_case(size="3b", layers=2, dtype="float32", batch=spread(1, 8), context=spread(16, 256),
                              arrivals=spread(1, 3), prompt=spread(1, 128), budget=128, decode=rng.randint(2, 4))
        if _cost(case) <= most and _tokens(case) <= 40000:
            return case


def _tokens(case):
    return sum(case["context"] + case["decode"] for _ in range(case["batch"])) + case["arrivals"] * case["prompt"]


# ------------------------------------------------------------------------------------------------ what a pass runs
def _lengths(most, count, unit):
    """``count`` lengths between a quarter of ``most`` and all of it, the first one ``most``; multiples of ``unit``."""
    return [max(unit, int(most * (1.0 - 0.75 * i / count)) // unit * unit) for i in range(count)]


def _plan(case):
    """``(lengths in the cache, prompt lengths, steps)``; a step is a list of ``(request, start, tokens, wants logits)`` with
    the running requests first.  A request's tokens are its context or prompt, then what it decodes."""
    there = _lengths(case["context"], case["batch"], PAGE)
    prompts = _lengths(case["prompt"], case["arrivals"], 1)
    at = there + [0] * len(prompts)
    running = list(range(len(there)))
    queue = list(range(len(there), len(at)))
    steps, decoded = [], 0
    while queue or decoded < case["decode"]:
        step = []
        if running and decoded < case["decode"]:
            step = [(r, at[r], 1, True) for r in running]
            decoded += 1
        room, through = case["budget"], []
        while queue and room > 0:
            r = queue[0]
            left = prompts[r - len(there)] - at[r]
            n = min(left, room)
            step.append((r, at[r], n, n == left))
            room -= n
            if n < left:
                at[r] += n
                break
            through.append(queue.pop(0))
        for r, start, n, _ in step:
            at[r] = start + n
        running = running + through
        steps.append(step)
    return there, prompts, steps


def _token_lists(case, seed):
    there, prompts, _ = _plan(case)
    vocab = SIZES[case["size"]][4]
    rng = np.random.default_rng(seed)
    return [rng.integers(0, vocab, n + case["decode"]).tolist() for n in there + prompts]


def _config(case):
    width, ff, heads, kv, vocab, tied = SIZES[case["size"]]
    if case["design"] == "qwen25vl":
        return {"architectures": ["Qwen2_5_VLForConditionalGeneration"], "model_type": "qwen2_5_vl", "hidden_size": width,
                "intermediate_size": ff, "num_hidden_layers": case["layers"], "num_attention_heads": heads,
                "num_key_value_heads": kv, "vocab_size": vocab, "tie_word_embeddings": tied, "rms_norm_eps": 1e-6,
                "rope_theta": 1000000.0, "max_position_embeddings": 32768, "use_sliding_window": False,
                "rope_scaling": {"type": "mrope", "mrope_section": [16, 24, 24]}}
    dense = {"kind": "dense", "ff": ff, "limit": 7.0} if case["design"] == "gogudra" else {"kind": "dense", "ff": ff}
    if case["design"] == "gogudra":
        mixers = {
            "gla": {"heads": heads, "dim": HEAD // 2, "vdim": HEAD, "tau": 16.0, "rank": 16},
            "lightning": {"heads": heads, "dim": HEAD, "vdim": HEAD,
                          "decay": [1.0 - 2.0 ** (-5.0 - 3.0 * i / max(1, heads - 1)) for i in range(heads)]},
            "attention": {"heads": heads, "kv_heads": kv, "dim": HEAD, "vdim": HEAD, "scale": HEAD ** -0.5,
                          "rot": {"base": 500000.0, "dims": HEAD // 2,
                                  "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}}}
        order = ("gla", "gla", "lightning", "attention")
        return {"architecture": "Gogudra", "width": width, "vocab": vocab, "norm": {"eps": 1e-6}, "logit_softcap": 30.0,
                "layers": [{"type": order[i % 4], "mixer": mixers[order[i % 4]], "mlp": dense} for i in range(case["layers"])]}
    part = ff // 8 // 16 * 16
    moe = {"kind": "moe", "expert": {"ff": part}, "shared": {"ff": 2 * part}, "router": {"experts": 32, "top": 6}}
    mixers = {
        "attention": {"heads": heads, "kv_heads": kv, "dim": HEAD, "vdim": HEAD, "scale": HEAD ** -0.5,
                      "rot": {"base": 1000000.0, "dims": HEAD // 2}},
        "attention_2": {"heads": heads, "kv_heads": kv, "dim": HEAD, "vdim": HEAD, "conv": 4, "mask": {"size": 1024},
                        "scale": HEAD ** -0.5, "rot": {"base": 10000.0, "dims": HEAD // 2, "scaling": {"factor": 4.0}}},
        "latent_attention": {"heads": heads, "dim": HEAD, "rot_dim": 64, "vdim": HEAD, "kv_rank": 192,
                             "scale": (HEAD + 64) ** -0.5,
                             "rot": {"base": 100000.0, "dims": 64,
                                     "scaling": {"factor": 8.0, "original": 8192, "fast": 16.0, "slow": 2.0}}}}
    order = ("attention", "attention_2", "latent_attention", "attention_2")
    return {"architecture": "Rofapel", "width": width, "vocab": vocab, "norm": {"eps": 1e-6}, "embedding": {"scale": 2.0},
            "layers": [{"type": order[i % 4], "mixer": mixers[order[i % 4]], "mlp": dense if i % 4 == 0 else moe}
                       for i in range(case["layers"])]}


def _draw_tensor(case, seed, name, shape):
    """A weight by its name, on the GPU: matrices N(0, 0.02) in the run's type, vectors in float32; gains around one (around
    zero where the design stores them so), routers and decays spread as trained ones are."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(zlib.crc32(f"{seed}:{name}".encode()))
    vector = len(shape) == 1 or name.endswith(".conv.weight")
    dtype = torch.float32 if vector or case["dtype"] == "float32" else torch.bfloat16
    mean, std = 0.0, 0.02
    leaf = name.split(".")
    if case["design"] == "qwen25vl":           # a residual sum that its layers change little by little
        if name.startswith("embed_tokens"):
            std = 0.3 if SIZES[case["size"]][5] else 1.0
        elif leaf[-2] in ("o_proj", "down_proj"):
            std = 0.005
    if name.endswith("router.weight"):
        std = 3.0 / math.sqrt(shape[1])        # logits with a spread of about 3: a few experts stand out
    elif name.endswith("a2.bias"):
        mean, std = 2.0, 1.0                   # gates that mostly keep
    elif name.endswith(".conv.weight"):
        std = 0.5
    elif name.endswith("sink.weight"):
        std = 1.0
    elif vector and any(k.endswith("norm") or k.endswith("layernorm") for k in leaf):
        mean = 1.0
    if leaf[-2] in ("norm1", "norm2") or (case["design"] != "qwen25vl" and name.startswith("final.norm")):
        mean = 0.0                             # stored around zero
    return torch.empty(tuple(shape), dtype=dtype, device="cuda").normal_(mean, std, generator=gen)


# ------------------------------------------------------------------------------------------------ the framework's side
def prepare(case, seed):
    if case["kind"] == "sample":
        return _prepare_sample(case, seed)
    from qwen25vl_lite_amd import EngineConfig, ModelRunner, build_model
    from qwen25vl_lite_amd.config import load_config
    from qwen25vl_lite_amd.engine.batch import StepEntry

    dtype = getattr(torch, case["dtype"])
    model = build_model(load_config(_config(case)), dtype, "cuda:0")
    expected = model.expected_tensors()
    for part, names in model.part_groups():
        tensors = {local: _draw_tensor(case, seed, name, expected[name].shape) for local, name in names.items()
                   if not (name == model.spec.head_name and model.spec.tie_word_embeddings)}
        if tensors:
            model.load_part(part, tensors)
    if model.spec.tie_word_embeddings:
        model.tie_head()

    there, prompts, steps = _plan(case)
    tokens = _token_lists(case, seed)
    page_need = sum((n + case["decode"]) // PAGE + 2 for n in there + prompts) + sum(n // PAGE for n in there)
    longest = max(len(t) for t in tokens)
    runner = ModelRunner(model, EngineConfig(
        num_blocks=page_need, block_size=PAGE, max_num_seqs=2 * len(there) + len(prompts),
        max_num_batched_tokens=max(4096, case["budget"] + len(there)), max_model_len=max(8192, longest),
        enable_prefix_cache=False, dtype=dtype, device="cuda:0", hip_graph=True))
    for r, n in enumerate(there):
        runner.admit(("kept", r))
    at = [0] * len(there)
    while any(a < n for a, n in zip(at, there)):        # what the running requests read before, a few thousand tokens a step
        entries, room = [], 4096
        for r, n in enumerate(there):
            take = min(n - at[r], room)
            if take > 0:
                entries.append(StepEntry(("kept", r), tokens[r][at[r]:at[r] + take], at[r]))
                at[r] += take
                room -= take
        runner.execute(entries)
    plan = [[StepEntry(r, tokens[r][start:start + n], start, [n - 1] if want else []) for r, start, n, want in step]
            for step in steps]
    return {"runner": runner, "kept": len(there), "new": len(prompts), "plan": plan}


def run(state):
    if "logits" in state:
        from qwen25vl_lite_amd.sampling.sampler import sample_rows
        return np.asarray(sample_rows(state["logits"], state["params"], state["previous"], state["generated"]))
    runner, kept = state["runner"], state["kept"]
    for r in range(kept):
        runner.fork(("kept", r), r)
    for r in range(kept, kept + state["new"]):
        runner.admit(r)
    outputs = []
    for entries in state["plan"]:
        outputs.append(runner.execute(entries).clone())    # a decode step's logits lie in a buffer that the next one fills
    for r in range(kept + state["new"]):
        runner.release(r)
    return outputs


def _prepare_sample(case, seed):
    from qwen25vl_lite_amd import SamplingParams

    rows, vocab = case["rows"], case["vocab"]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    # a language model's logits: a wide bell, and some dozens of tokens well above it
    logits = torch.empty(rows, vocab, device="cuda").normal_(0.0, 2.0, generator=gen)
    likely = torch.randint(0, vocab, (rows, 40), device="cuda", generator=gen)
    logits.scatter_add_(1, likely, torch.empty(rows, 40, device="cuda").normal_(7.0, 3.0, generator=gen))
    rng = np.random.default_rng(seed)
    kinds = [dict(temperature=0.0), dict(temperature=0.7, top_p=0.9),
             dict(temperature=1.0, top_k=50, top_p=0.95, repetition_penalty=1.05, frequency_penalty=0.1),
             dict(temperature=0.8, min_p=0.05)]
    params, previous, generated = [], [], []
    for i in range(rows):
        params.append(SamplingParams(seed=int(rng.integers(1 << 30)), **kinds[i % 4]))
        generated.append(int(rng.integers(1, 400)))
        previous.append(rng.integers(0, vocab, generated[-1]).tolist())
    return {"logits": logits, "params": params, "previous": previous, "generated": generated}


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def _layer_matrices(case, i):
    """``(values of the layer's matrices that every token uses, (experts, top, values an expert), value heads' cache per token)``."""
    width, ff, heads, kv, _, _ = SIZES[case["size"]]
    if case["design"] == "qwen25vl":
        return width * (heads + 2 * kv) * HEAD + heads * HEAD * width + 3 * width * ff, None, 2 * kv * HEAD
    if case["design"] == "gogudra":
        kind = ("gla", "gla", "lightning", "attention")[i % 4]
        d = {"gla": heads * HEAD // 2, "lightning": heads * HEAD, "attention": 0}[kind]
        mixer = (width * (heads + kv) * HEAD + heads * HEAD * width if kind == "attention"
                 else 2 * width * d + 3 * width * heads * HEAD)
        return mixer + 3 * width * ff, None, 2 * kv * HEAD if kind == "attention" else 0
    part = ff // 8 // 16 * 16
    kind = ("attention", "attention_2", "latent", "attention_2")[i % 4]
    if kind == "latent":
        mixer = width * heads * (HEAD + 64) + width * 256 + 2 * heads * HEAD * 192 + heads * HEAD * width
        cache = 256
    else:
        mixer = width * (heads + (2 if kind == "attention" else 1) * kv) * HEAD + heads * HEAD * width
        cache = 2 * kv * HEAD
    if i % 4 == 0:
        return mixer + 3 * width * ff, None, cache
    return mixer + 3 * width * 2 * part + 32 * width, (32, 6, 3 * width * part), cache


def _state_values(case, i):
    heads = SIZES[case["size"]][2]
    if case["design"] == "gogudra" and i % 4 < 3:
        return heads * HEAD * (HEAD // 2 if i % 4 < 2 else HEAD)
    return 0


def work(case):
    if case["kind"] == "sample":
        return {"bytes": 4.0 * case["rows"] * case["vocab"], "flops": 6.0 * case["rows"] * case["vocab"]}
    width, _, heads, _, vocab, _ = SIZES[case["size"]]
    size = 4 if case["dtype"] == "float32" else 2
    read = written = flops = 0.0
    for step in _plan(case)[2]:
        n = sum(t for _, _, t, _ in step)
        wants = sum(w for _, _, _, w in step)
        pairs = sum(t * s + t * (t + 1) / 2 for _, s, t, _ in step)        # (token, key it sees)
        cached = sum(s for _, s, _, _ in step)
        for i in range(case["layers"]):
            plain, experts, cache = _layer_matrices(case, i)
            read += plain * size + cached * cache * size
            written += n * cache * size
            flops += 2.0 * n * plain
            if experts:
                count, top, values = experts
                read += count * (1.0 - (1.0 - top / count) ** n) * values * size
                flops += 2.0 * n * top * values
            if cache:
                flops += 4.0 * heads * HEAD * pairs
            if _state_values(case, i):
                read += len(step) * _state_values(case, i) * 4
                written += len(step) * _state_values(case, i) * 4
                flops += 4.0 * n * _state_values(case, i)
        read += n * width * size + (vocab * width * size if wants else 0)
        written += wants * vocab * 4
        flops += 2.0 * wants * vocab * width
    return {"bytes": read + written, "flops": flops}


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def tolerance(case):
    if case["kind"] == "sample":
        return {"rel": 0.0, "differ": 0.01}
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 1e-4}      # measured against 64 bits: 2e-6 to 4e-6
    # bfloat16 storage leaves the logits 0.4 to 0.9 per cent from 64-bit arithmetic here; a token whose sixth and seventh
    # experts are close may change one for the other
    return {"rel": 0.02, "max": 0.8 if case["design"] == "rofapel" else 0.3}


# ------------------------------------------------------------------------------------------------ the same in 64 bits
def exact(case, seed):
    """The same logits with plain torch in float64, whole sequences at a time."""
    if case["kind"] == "sample":
        return None
    there, prompts, steps = _plan(case)
    tokens = _token_lists(case, seed)
    wanted = [[] for _ in tokens]                       # per request the places whose logits are asked for
    reach = [0] * len(tokens)
    for step in steps:
        for r, start, n, want in step:
            reach[r] = start + n
            if want:
                wanted[r].append(start + n - 1)
    seqs = [torch.tensor(t[:n], device="cuda") for t, n in zip(tokens, reach)]
    with torch.no_grad():
        logits = _Exact(case, seed, seqs).logits(wanted)
    place = {}
    for r, places in enumerate(wanted):
        for p in places:
            place[r, p] = len(place)
    return [logits[[place[r, start + n - 1] for r, start, n, want in step if want]] for step in steps]


class _Exact:
    def __init__(self, case, seed, seqs):
        self.case, self.seed, self.seqs = case, seed, seqs
        self.width, self.ff, self.heads, self.kv, self.vocab, self.tied = SIZES[case["size"]]
        self.ends = np.cumsum([0] + [len(s) for s in seqs]).tolist()
        self.pos = torch.cat([torch.arange(len(s), device="cuda") for s in seqs]).double()

    def w(self, name, *shape):
        return _draw_tensor(self.case, self.seed, name, shape).double()

    def product(self, x, name, rows, cols):
        """``x @ W.T``, some thousand of the weight's rows at a time."""
        weight = _draw_tensor(self.case, self.seed, name, (rows, cols))
        return torch.cat([x @ part.double().t() for part in weight.split(8192)], dim=1)

    def each(self, fn, *xs):
        """``fn`` for the rows of every request by themselves."""
        return torch.cat([fn(*(x[a:b] for x in xs)) for a, b in zip(self.ends, self.ends[1:])])

    def norm(self, x, gain, eps=1e-6):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * gain

    def rotate(self, x, freqs, amplitude=1.0, neighbours=False):
        half = freqs.shape[0]
        angle = self.pos[:, None, None] * freqs
        c, s = torch.cos(angle) * amplitude, torch.sin(angle) * amplitude
        first = slice(0, 2 * half, 2) if neighbours else slice(0, half)
        second = slice(1, 2 * half, 2) if neighbours else slice(half, 2 * half)
        out = x.clone()
        out[..., first] = x[..., first] * c - x[..., second] * s
        out[..., second] = x[..., second] * c + x[..., first] * s
        return out

    def attend(self, q, k, v, scale, window=None, sink=None):
        """Causal softmax attention, ``[T, heads, d]`` over ``[T, key heads, d]``, a thousand queries at a time."""
        per = q.shape[1] // k.shape[1]

        def one(q, k, v):
            k, v = k.transpose(0, 1), v.transpose(0, 1)                       # [G, T, d]
            out = []
            for lo in range(0, len(q), 1024):
                hi = min(len(q), lo + 1024)
                i = torch.arange(lo, hi, device="cuda")[:, None]
                j = torch.arange(hi, device="cuda")[None]
                hidden = (j > i) if window is None else (j > i) | (i - j >= window)
                heads = []
                for h in range(q.shape[1]):
                    s = (q[lo:hi, h] @ k[h // per, :hi].t() * scale).masked_fill_(hidden, -math.inf)
                    top = s.amax(-1, keepdim=True)
                    e = torch.exp(s - top)
                    total = e.sum(-1, keepdim=True)
                    if sink is not None:
                        total = total + torch.exp(sink[h] - top)
                    heads.append(e @ v[h // per, :hi] / total)
                out.append(torch.stack(heads, 1))
            return torch.cat(out)
        return self.each(one, q, k, v)

    # -------------------------------------------------------------------------------------------- the models
    def logits(self, wanted):
        plain = self.case["design"] == "qwen25vl"
        first = {"qwen25vl": "embed_tokens.weight"}.get(self.case["design"], "embed.weight")
        table = _draw_tensor(self.case, self.seed, first, (self.vocab, self.width))
        x = table[torch.cat(self.seqs)].double() * (2.0 if self.case["design"] == "rofapel" else 1.0)
        for i in range(self.case["layers"]):
            x = getattr(self, "layer_" + self.case["design"])(i, x)
        rows = [a + p for a, places in zip(self.ends, wanted) for p in places]
        gain = self.w("norm.weight" if plain else "final.norm.weight", self.width)
        x = self.norm(x[rows], gain if plain else 1.0 + gain)
        if (plain and self.tied) or self.case["design"] == "gogudra":
            y = torch.cat([x @ part.double().t() for part in table.split(8192)], dim=1)
        else:
            y = self.product(x, "lm_head.weight" if plain else "head.weight", self.vocab, self.width)
        return torch.tanh(y / 30.0) * 30.0 if self.case["design"] == "gogudra" else y

    def feed_forward(self, x, prefix, ff, act):
        out = torch.zeros_like(x)
        gate, up, down = (_draw_tensor(self.case, self.seed, f"{prefix}{n}.weight", s) for n, s in
                          zip(self.ff_names, ((ff, self.width), (ff, self.width), (self.width, ff))))
        for lo in range(0, ff, 4096):                    # some of the inner channels at a time
            s = slice(lo, min(ff, lo + 4096))
            out += act(x @ gate[s].double().t(), x @ up[s].double().t()) @ down[:, s].double().t()
        return out

    @property
    def ff_names(self):
        return ("gate_proj", "up_proj", "down_proj") if self.case["design"] == "qwen25vl" else ("gate", "up", "down")

    def layer_qwen25vl(self, i, x):
        p, n, nq, nk = f"layers.{i}.", len(x), self.heads * HEAD, self.kv * HEAD
        h = self.norm(x, self.w(p + "input_layernorm.weight", self.width))
        q, k, v = (self.product(h, f"{p}self_attn.{s}_proj.weight", rows, self.width)
                   + self.w(f"{p}self_attn.{s}_proj.bias", rows) for s, rows in (("q", nq), ("k", nk), ("v", nk)))
        freqs = 1000000.0 ** (-torch.arange(0, HEAD, 2, device="cuda").double() / HEAD)
        q, k = self.rotate(q.view(n, -1, HEAD), freqs), self.rotate(k.view(n, -1, HEAD), freqs)
        o = self.attend(q, k, v.view(n, -1, HEAD), HEAD ** -0.5)
        x = x + self.product(o.reshape(n, nq), p + "self_attn.o_proj.weight", self.width, nq)
        h = self.norm(x, self.w(p + "post_attention_layernorm.weight", self.width))
        return x + self.feed_forward(h, p + "mlp.", self.ff, lambda g, u: g * torch.sigmoid(g) * u)

    def layer_gogudra(self, i, x):
        p, n, kind = f"l{i}.", len(x), ("gla", "gla", "lightning", "attention")[i % 4]
        h = self.norm(x, 1.0 + self.w(p + "norm1.weight", self.width))
        y = self.feed_forward(h, p + "mlp.", self.ff,
                              lambda g, u: (lambda g, u: g * torch.sigmoid(1.702 * g) * (u + 1.0))(g.clamp(max=7.0), u.clamp(-7.0, 7.0)))
        m, nv = p + "mix.", self.heads * HEAD
        silu = lambda z: z * torch.sigmoid(z)
        if kind == "attention":
            q = self.product(h, m + "q.weight", nv, self.width).view(n, -1, HEAD)
            v = self.product(h, m + "k.weight", self.kv * HEAD, self.width).view(n, -1, HEAD)
            freqs = 500000.0 ** (-torch.arange(0, HEAD // 2, 2, device="cuda").double() / (HEAD // 2))
            wave = 2.0 * math.pi / freqs
            blend = ((8192 / wave - 1.0) / 3.0).clamp(0.0, 1.0)               # long wavelengths slowed, short ones kept
            freqs = (1.0 - blend) * freqs / 8.0 + blend * freqs
            q = self.rotate(self.norm(q, self.w(m + "q.norm.weight", HEAD)), freqs, neighbours=True)
            k = self.rotate(self.norm(v, self.w(m + "k.norm.weight", HEAD)), freqs, neighbours=True)
            o = self.attend(q, k, v, HEAD ** -0.5)
            o = (o * torch.sigmoid(self.product(h, m + "g.weight", self.heads, self.width))[:, :, None]).reshape(n, nv)
        else:
            d = HEAD // 2 if kind == "gla" else HEAD
            q, k, v = (self.product(h, f"{m}{s}.weight", rows, self.width) for s, rows in
                       (("q", self.heads * d), ("k", self.heads * d), ("v", nv)))
            if kind == "gla":
                q = q * d ** -0.5
                z = self.product(self.product(h, m + "a1.weight", 16, self.width), m + "a2.weight", self.heads * d, 16)
                decay = torch.exp(torch.nn.functional.logsigmoid(z + self.w(m + "a2.bias", self.heads * d)) / 16.0)
            else:
                q, k, v = silu(q), silu(k), silu(v)
                per_head = torch.tensor([1.0 - 2.0 ** (-5.0 - 3.0 * j / max(1, self.heads - 1)) for j in range(self.heads)],
                                        dtype=torch.float32, device="cuda").double()
                decay = per_head[:, None].expand(self.heads, d).reshape(1, -1).expand(n, -1)
            o = self.each(self.scan, *(t.reshape(n, self.heads, -1) for t in (q, k, v, decay)))
            gate = self.product(h, m + "g.weight", nv, self.width)
            if kind == "gla":
                o = self.norm(o, self.w(m + "norm.weight", HEAD)).reshape(n, nv) * silu(gate)
            else:
                o = self.norm(o.reshape(n, nv), self.w(m + "norm.weight", nv)) * torch.sigmoid(gate)
        return x + y + self.product(o, m + "o.weight", self.width, nv)

    @staticmethod
    def scan(q, k, v, decay):
        """``S <- diag(decay) S + k v^T, o = S^T q`` token after token, all heads at once."""
        state = torch.zeros(q.shape[1], q.shape[2], v.shape[2], dtype=q.dtype, device=q.device)
        out = torch.empty_like(v)
        for t in range(len(q)):
            state = torch.baddbmm(decay[t][:, :, None] * state, k[t][:, :, None], v[t][:, None, :])
            out[t] = torch.bmm(q[t][:, None, :], state)[:, 0]
        return out

    def layer_rofapel(self, i, x):
        p, n, kind = f"l{i}.", len(x), ("attention", "attention_2", "latent", "attention_2")[i % 4]
        m, nv, part = p + "mix.", self.heads * HEAD, self.ff // 8 // 16 * 16
        h = self.norm(x, 1.0 + self.w(p + "norm1.weight", self.width))
        powers = lambda base, dims: base ** (-torch.arange(0, dims, 2, device="cuda").double() / dims)
        if kind == "latent":
            q = self.product(h, m + "q.weight", self.heads * 192, self.width).view(n, -1, 192)
            down = self.product(h, m + "dkv.weight", 256, self.width)
            c = self.norm(down[:, :192], self.w(m + "dkv.norm.weight", 192))
            turn = lambda turns: 64 * math.log(8192 / (2.0 * math.pi * turns)) / (2.0 * math.log(100000.0))
            lo, hi = max(math.floor(turn(16.0)), 0), min(math.ceil(turn(2.0)), 63)
            ramp = ((torch.arange(32, device="cuda").double() - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
            freqs = powers(100000.0, 64)
            freqs, amp = freqs / 8.0 * ramp + freqs * (1.0 - ramp), 0.1 * math.log(8.0) + 1.0
            turned = self.rotate(down[:, None, 192:], freqs, amp, neighbours=True)
            q = torch.cat([q[..., :HEAD], self.rotate(q[..., HEAD:], freqs, amp, neighbours=True)], -1)
            k = self.product(c, m + "uk.weight", nv, 192).view(n, -1, HEAD)
            v = self.product(c, m + "uv.weight", nv, 192).view(n, -1, HEAD)
            o = self.attend(q, torch.cat([k, turned.expand(n, self.heads, 64)], -1), v, 192 ** -0.5).reshape(n, nv)
        else:
            q, k = (self.product(h, f"{m}{s}.weight", rows, self.width) for s, rows in (("q", nv), ("k", self.kv * HEAD)))
            freqs, sink, window = powers(1000000.0, HEAD // 2), None, None
            if kind == "attention":
                v = self.product(h, m + "v.weight", self.kv * HEAD, self.width)
                q = self.norm(q, self.w(m + "q.norm.weight", nv)).view(n, -1, HEAD)
                k = self.norm(k, self.w(m + "k.norm.weight", self.kv * HEAD)).view(n, -1, HEAD)
            else:
                def taps(u, w):
                    pad = torch.cat([torch.zeros(3, u.shape[1], dtype=u.dtype, device=u.device), u])
                    return sum(pad[j:j + len(u)] * w[:, j] for j in range(4))
                wq, wk = self.w(m + "q.conv.weight", nv, 4), self.w(m + "k.conv.weight", self.kv * HEAD, 4)
                q, k = self.each(lambda u: taps(u, wq), q), self.each(lambda u: taps(u, wk), k)
                v, freqs, window = k, powers(10000.0, HEAD // 2) / 4.0, 1024
                sink = self.w(m + "sink.weight", self.heads)
                q = self.norm(q.view(n, -1, HEAD), self.w(m + "q.norm.weight", HEAD))
                k = self.norm(k.view(n, -1, HEAD), self.w(m + "k.norm.weight", HEAD))
            o = self.attend(self.rotate(q, freqs), self.rotate(k, freqs), v.view(n, -1, HEAD), HEAD ** -0.5, window, sink)
            gate = torch.sigmoid(self.product(h, m + "g.weight", self.heads, self.width))
            o = (o * gate[:, :, None]).reshape(n, nv)
        h = self.norm(x, 1.0 + self.w(p + "norm2.weight", self.width))       # both sublayers read the layer's input
        x = x + self.product(o, m + "o.weight", self.width, nv)
        act = lambda g, u: g * torch.sigmoid(g) * u
        f = p + "mlp."
        if i % 4 == 0:
            return x + self.feed_forward(h, f, self.ff, act)
        z = self.product(h, f + "router.weight", 32, self.width) + self.w(f + "router.bias", 32)
        top, chosen = z.topk(6, -1)
        share = torch.softmax(top, -1)
        y = self.feed_forward(h, f + "shared.", 2 * part, act)
        for e in range(32):
            rows, column = (chosen == e).nonzero(as_tuple=True)
            if len(rows):
                y[rows] += share[rows, column][:, None] * self.feed_forward(h[rows], f"{f}e{e}.", part, act)
        return x + y
