"""Rules that choose a kernel by sizes, and what the sampler is handed: what can be checked without a GPU."""

import numpy as np
import pytest
import torch


@pytest.mark.parametrize("cus", [32, 64, 256])
@pytest.mark.parametrize("rows", [1, 8, 9, 64])
def test_products_are_cut_where_the_kernel_takes_the_cut(cus, rows, monkeypatch):
    """What takes_split accepts, the kernel behind it divides into ranges, on a device of any number of compute units (a part of
    one, say): the inner size may be as long as its blocks can keep."""
    from qwen25vl_lite_amd.ops import skinny
    monkeypatch.setattr(skinny, "_compute_units", lambda device: cus)
    taken = 0
    for k in [8, 4096, 4104, 2048 * cus - 8, 2048 * cus, 2048 * cus + 8, 4096 * cus, 4096 * cus + 8, 8192 * cus]:
        if skinny.takes_split(rows, k, torch.empty((3, k), dtype=torch.bfloat16)):
            taken += 1
            assert skinny._ranges(rows, 3, k, cus) > 0, k
    assert taken >= 5


def test_sampler_takes_token_ids_of_any_kind():
    """Lists of Python's and numpy's integers, 0-d tensors, arrays and tensors of one id each; what is no id is refused."""
    from qwen25vl_lite_amd.sampling.sampler import _int32_ids
    for flat in ([3, 4], [np.int64(3), np.uint8(4)], list(torch.tensor([3, 4])), list(torch.tensor([[3], [4]])),
                 list(np.array([[3], [4]], np.int64)), ["3", 4]):
        got = _int32_ids(flat)
        assert got.dtype == np.int32 and got.tolist() == [3, 4], flat
    assert _int32_ids([]).tolist() == [0]
    for flat, error in (([1 << 40], OverflowError), ([np.int64(1 << 40)], OverflowError), ([None], TypeError),
                        (list(torch.tensor([[3, 4], [5, 6]])), (RuntimeError, TypeError, ValueError))):
        with pytest.raises(error):
            _int32_ids(flat)


def test_sampler_settings_gathered_by_native_code():
    """The words that go to the device are those that Python's loop makes, at any settings, number of ids and room; what is
    not of the usual kind is left to that loop."""
    from qwen25vl_lite_amd.sampling import SamplingParams
    from qwen25vl_lite_amd.sampling import sampler as S
    kinds = [dict(temperature=0.0), dict(temperature=0.7, top_p=0.9, seed=3), dict(temperature=1, top_k=50, repetition_penalty=1.05, seed=-9),
             dict(temperature=0.8, min_p=0.05, seed=2 ** 40 + 7), dict(temperature=0.0, presence_penalty=0.5), dict(temperature=2.0, top_k=0, seed=1)]
    params = [SamplingParams(**k) for k in kinds]
    prev = [[5], (1, 2), [2 ** 30 - 1, 0, 2 ** 30, -1, 2 ** 31 - 1], [], list(range(300)), []]
    steps = [1, 2, 5, 0, 300, 7]
    rows, ids = np.zeros(len(params), S._ROW), []
    for i, p in enumerate(params):
        begin = len(ids)
        if p.repetition_penalty != 1.0 or p.presence_penalty != 0.0 or p.frequency_penalty != 0.0:
            ids.extend(prev[i])
        seeded = p.temperature > 0
        rows[i] = (p.temperature, p.top_p, p.min_p, 0.0, p.repetition_penalty, p.presence_penalty, p.frequency_penalty, p.top_k or -1, begin,
                   len(ids), (p.seed + steps[i]) & 0xffffffff if seeded else 0, seeded)
    want = np.concatenate([rows.view(np.int32), np.asarray(ids, np.int32)])
    host = torch.full((want.size + 3,), 77, dtype=torch.int32)
    words, flags = S._gather(params, prev, steps, 100, host)
    assert words == want.size and host[:words].tolist() == want.tolist() and host[words:].tolist() == [77] * 3
    assert list(flags) == [1, 1, 1, 1]
    small = torch.full((80,), 77, dtype=torch.int32)
    assert S._gather(params, prev, steps, 100, small[:76])[0] == -want.size and small[76:].tolist() == [77] * 4
    assert S._gather(params[:1], prev[:1], steps[:1], 100, host)[0] == 13 and host[12] == 0        # no ids: one zero
    for odd in (dict(params=[SamplingParams(temperature=0.5)]), dict(params=[SamplingParams(temperature="1")]), dict(params=[None]),
                dict(params=[SamplingParams(temperature=1.0, seed=2 ** 70)]), dict(prev=[np.array([3])]), dict(prev=[[2 ** 31]]),
                dict(prev=[[np.int64(3)]]), dict(prev=[[True]]), dict(steps=[np.int64(1)]), dict(prev=[]), dict(steps=np.array([1]))):
        call = dict(params=[SamplingParams(temperature=1.0, seed=4, presence_penalty=0.1)], prev=[[3]], steps=[1])
        assert S._gather(call["params"], call["prev"], call["steps"], 100, host)[0] == 13
        call.update(odd)
        assert S._gather(call["params"], call["prev"], call["steps"], 100, host)[0] == -1, odd


@pytest.mark.parametrize("m, n, k, units, ranges", [
    (1031, 2048, 2048, 128, 3), (1031, 2048, 2048, 256, 1), (281, 2048, 2048, 256, 4), (281, 2048, 11008, 256, 5), (512, 3584, 3584, 256, 2),
    (1600, 3584, 18944, 256, 2), (2048, 3584, 18944, 256, 2), (3200, 3584, 18944, 256, 1), (700, 8192, 29568, 256, 5),
    (200, 2560, 2048, 64, 3), (300, 4608, 3584, 32, 1), (65, 64, 32, 256, 1), (5000, 8192, 8192, 304, 1)])
def test_ranges_of_the_inner_size_do_not_follow_the_tiles_shape(m, n, k, units, ranges):
    """How many ranges a product is cut into decides the order of its sums and whether they stay in float32: by the four
    shapes' estimate on any number of compute units, as these counts were before there were more shapes."""
    import ctypes

    from qwen25vl_lite_amd.ops.kernels import _fn
    assert _fn("gemm_tile", "qvl_gemm_tile_splits", [ctypes.c_int] * 4)(m, n, k, units) == ranges


def test_a_steps_lists_are_not_made_inside_a_graph(monkeypatch):
    """Their way to the device is by host memory that another list takes later: a recorded copy would read that one's numbers."""
    from qwen25vl_lite_amd.ops import attention_mfma, kernels, linear_attention
    lists = np.arange(5, dtype=np.int32)
    assert kernels.int32_to_device(lists, "cpu").tolist() == lists.tolist()
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    assert kernels.int32_to_device(lists, "cpu").tolist() == lists.tolist()
    for device in ("cuda:0", torch.device("cuda")):
        with pytest.raises(kernels.KernelError, match="captured"):
            kernels.int32_to_device(lists, device)
        with pytest.raises(kernels.KernelError, match="captured"):
            linear_attention.plan_chunks([0, 7, 9], device)

        class Step:
            derived, cu_q_host, ctx_len_host = {}, [0, 7, 9], [7, 2]
        with pytest.raises(kernels.KernelError, match="captured"):
            attention_mfma._step_tiles(Step, 4, 1, device)
        assert not Step.derived


@pytest.mark.parametrize("qlens, lens, group, nkv, window", [([2048], [2048], 7, 4, 0), ([512], [8192], 7, 4, 0), ([1], [40000], 8, 1, 0),
                                                             ([700, 1, 33], [3000, 9000, 33], 1, 6, 0), ([300, 0, 90], [5000, 7, 90], 5, 8, 1000),
                                                             ([1], [1], 1, 16, 0), ([20000], [30000], 16, 2, 0),
                                                             ([300, 5, 0, 129], [300, 400, 9, 200], 7, 3, 0)])
@pytest.mark.parametrize("places, groups, wide", [(512, 1, False), (256, 2, False), (512, 1, True), (13, 1, False)])
def test_walks_of_prompt_portions(qlens, lens, group, nkv, window, places, groups, wide):
    """Every run of column tiles of every head has its key blocks once, in parts that follow each other, longest first; the parts of
    cut walks have places of their own for their results; workgroups there are for all, and with few walks each has less than the longest walk."""
    from qwen25vl_lite_amd.ops import attention_mfma as attn
    cu = np.concatenate([[0], np.cumsum(qlens)])
    defines = attn.block_defines(128, wide)
    plan = attn.plan_walks(cu, lens, group, nkv, window, places, groups, defines)
    cols, per_head = 16 * attn.block_tiles(128, wide), 8 % nkv == 0
    heads = 1 if per_head else nkv
    walks = {}
    for req, cb, head, first, last, packed, slot, counter in plan.items.tolist():
        walks.setdefault((req, cb, head), []).append((packed & 0xffff, packed >> 16, first, last, slot, counter))
    want = {(r, cb, h) for r, q in enumerate(qlens) for cb in range(-(-q * group // cols)) for h in range(heads)}
    assert set(walks) == want
    slots, counters = [], []
    for (r, cb, _), parts in walks.items():
        parts.sort()
        before = lens[r] - qlens[r]
        lo = max(0, before + cb * cols // group - window + 1) if window else 0
        hi = before + min((cb * cols + cols - 1) // group, qlens[r] - 1)
        assert [p[0] for p in parts] == list(range(len(parts))) and {p[1] for p in parts} == {len(parts)}
        assert parts[0][2] == lo >> 5 and parts[-1][3] == hi >> 5
        assert all(a[3] + 1 == b[2] for a, b in zip(parts, parts[1:])) and all(p[2] <= p[3] for p in parts)
        if len(parts) > 1:
            slots += list(range(parts[0][4], parts[0][4] + len(parts)))
            counters.append(parts[0][5])
            assert len({p[4] for p in parts}) == len({p[5] for p in parts}) == 1
    assert sorted(slots) == list(range(len(slots))) and sorted(counters) == list(range(len(counters)))
    assert plan.partials == len(slots) * (nkv if per_head else 1)
    assert (plan.head_slots, plan.head_walks) == ((len(slots), len(counters)) if per_head else (0, 0))
    n = plan.items[:, 4] - plan.items[:, 3]
    assert (np.diff(n) <= 0).all()
    most = max(8 // nkv, places // 8 * 8 // nkv) if per_head else places
    assert plan.places == min(most, len(plan.items))
    # the workgroups launched reach every place of every head, and no more than eight beyond
    assert plan.grid >= plan.places * (nkv if per_head else 1) > plan.grid - 8
    if len(want) * 4 < most and n.max() >= 64:
        assert counters


@pytest.mark.parametrize("requests", [1, 63, 64, 150])
def test_runs_of_column_tiles_counted_by_integers_and_by_arrays(requests):
    from types import SimpleNamespace
    from qwen25vl_lite_amd.ops import attention_mfma as attn
    assert 63 < attn.MANY_REQUESTS <= 64
    rng = np.random.default_rng(requests)
    q = rng.integers(0, 300, requests)
    ctx = q + rng.integers(0, 4000, requests)
    cu = np.concatenate([[0], np.cumsum(q)]).tolist()
    for only in (None, tuple(int(x) for x in rng.integers(0, 2, requests))):
        step = SimpleNamespace(cu_q_host=cu, ctx_len_host=ctx.tolist(), derived={})
        for group, tile_ct in ((1, 1), (7, 8), (3, 12)):
            entries = [-(-int(n) * group // (16 * tile_ct)) * (only is None or only[i]) for i, n in enumerate(q)]
            assert attn._count_tiles(step, group, tile_ct, only) == sum(entries)
            assert attn._walk_blocks(step, group, tile_ct, only) == sum(
                e * max(1, (int(c) - int(n) // 2 + 31) // 32) for e, n, c in zip(entries, q, ctx))


def test_whole_walks_are_listed_longest_first():
    """The lists are made by counting; here once more by comparing: those of one length stay as they come."""
    from qwen25vl_lite_amd.ops import attention_mfma as attn
    rng = np.random.default_rng(5)
    for _ in range(20):
        q = rng.integers(1, 400, rng.integers(1, 40))
        ctx = q + rng.integers(0, 6000, len(q))
        group, nkv, places = int(rng.integers(1, 9)), int(rng.choice([2, 3, 8])), int(rng.choice([16, 100, 512]))
        plan = attn.plan_walks(np.concatenate([[0], np.cumsum(q)]), ctx, group, nkv, 0, places, 1, {"HD": 128}, cut=False)
        heads = 1 if 8 % nkv == 0 else nkv
        walks = [(r, cb, h, 0, (int(ctx[r]) - int(q[r]) + min((128 * cb + 127) // group, int(q[r]) - 1)) >> 5)
                 for r in range(len(q)) for cb in range(-(-int(q[r]) * group // 128)) for h in range(heads)]
        assert [tuple(i[:5]) for i in plan.items.tolist()] == sorted(walks, key=lambda w: -w[4]) and plan.partials == 0


@pytest.mark.parametrize("bad", [dict(lens=[3]), dict(groups=3), dict(nkv=0), dict(places=0)])
def test_walks_that_cannot_be_listed(bad):
    from qwen25vl_lite_amd.ops import attention_mfma as attn, kernels
    kw = {**dict(lens=[9], nkv=2, places=16, groups=1), **bad}
    with pytest.raises(kernels.KernelError):
        attn.plan_walks([0, 4], kw["lens"], 2, kw["nkv"], 0, kw["places"], kw["groups"], {"HD": 128})


@pytest.mark.parametrize("nq, nkv, hd, rows, keys", [(28, 4, 128, 200, 2048), (16, 4, 256, 160, 512), (64, 8, 128, 96, 1024), (9, 3, 96, 256, 512),
                                                     (64, 1, 64, 200, 2048), (64, 1, 64, 600, 2048)])
def test_walks_of_lengths_that_nobody_knows_stay_whole(nq, nkv, hd, rows, keys, monkeypatch):
    """A step captured for contexts of up to some length: its walks, where known ones would be cut, by two wave groups only where each has a
    workgroup to itself."""
    from types import SimpleNamespace
    from qwen25vl_lite_amd.ops import attention_mfma as attn
    monkeypatch.setattr(attn, "_work_queue", lambda device: (None, 256))
    step = SimpleNamespace(cu_q_host=list(range(rows + 1)), ctx_len_host=[keys] * rows, lengths_known=False, derived={})
    wide, groups, _, plan, _ = attn._step_walks(step, nq // nkv, nkv, hd, 0, "cpu")
    assert plan.partials == 0 and len(plan.items) == rows * (1 if 8 % nkv == 0 else nkv)
    assert groups == (2 if not wide and hd <= 128 and rows * nkv <= 512 else 1)
    if rows * nkv in (800, 640, 768):
        known = SimpleNamespace(**{**vars(step), "lengths_known": True, "derived": {}})
        assert attn._step_walks(known, nq // nkv, nkv, hd, 0, "cpu")[3].partials > 0


@pytest.mark.parametrize("ranges", range(5))
@pytest.mark.parametrize("k", [512, 2048, 3584, 8192])
def test_products_that_are_cut_stay_cut(k, ranges):
    """The projection with the rotation inside sums in one chain: it takes only what has one chain anyway."""
    from qwen25vl_lite_amd.ops import tile
    x, w = torch.empty(300, k, dtype=torch.bfloat16), torch.empty(6 * 128, k, dtype=torch.bfloat16)
    assert tile.prefers_heads(x, w, ranges, 128, 64) == (ranges == 1)


def test_slices_are_asked_for_without_the_library(monkeypatch):
    """Every layer of a step asks: by the kernel's own rule, but in plain integers."""
    import ctypes
    from qwen25vl_lite_amd.ops import kernels, skinny
    rule = kernels._fn("gemm_slice", "qvl_gemm_slice_takes", [ctypes.c_int] * 4)
    for m in (0, 1, 64, 65):
        for k in (0, 8, 12, 4088, 4096, 4104):
            for n in (0, 2, 3, 8190, 8192, 8194, 9728):
                for cus in (1, 256, 304):
                    assert skinny._slice_fits(m, k, n, cus) == bool(rule(m, n, k, cus)), (m, k, n, cus)
    asked = []
    monkeypatch.setattr(skinny, "_fn", lambda *a, **kw: asked.append(a))
    monkeypatch.setattr(skinny, "_compute_units", lambda device: 256)
    w = torch.empty(256, 512, dtype=torch.bfloat16)
    for weight, head, half, cache, want in ((w, 64, 32, torch.bfloat16, True), (w, 64, 32, None, True), (w, 64, 16, None, False), (w.float(), 64, 32, None, False),
                                            (w, 64, 32, torch.float32, False), (w[:, 1:], 64, 32, None, False), (w.t(), 64, 32, None, False)):
        assert skinny.takes_slice(5, weight.shape[1], weight, head, half, cache) == want
    assert not asked


def test_no_wave_routes_two_tokens_in_one_launch():
    """Routing and listing in one block of sixteen waves: a token for each of half of them at most."""
    from qwen25vl_lite_amd.ops import kernels
    assert 1 <= kernels._fn("moe", "qvl_moe_route_rows", [])() <= 8


def test_which_rows_of_the_stacked_projection_are_cut():
    """17 to 48 rows at any size, up to 64 of large weights beyond the inner size that the kernel with the rotation inside keeps in one
    pass."""
    from qwen25vl_lite_amd.ops import skinny
    from qwen25vl_lite_amd.parts import attention

    def cut(n, k):
        return [m for m in range(1, 70) if attention._splits(m, n, k)]
    for n, k in ((2560, 2048), (4608, 3584), (40960, 4096), (512, 4608), (7168, 5120), (1280, 8192), (5119, 8192)):
        assert cut(n, k) == list(range(17, 49)), (n, k)
    for n, k in ((10240, 4104), (5120, 8192), (10240, 6144), (10240, 8192), (18432, 16384)):
        assert cut(n, k) == list(range(17, 65)), (n, k)
    for k in (4104, 8192):        # what ran there before is the library's product, not the fused kernel
        assert not any(skinny.takes_resident(m, k, torch.empty((10240, k), dtype=torch.bfloat16, device="meta")) for m in range(33, 65))


def test_sampler_settings_of_rows_without_a_seed():
    """Rows that draw without a seed are gathered with the others and marked, whatever their place among the steps."""
    import ctypes

    from qwen25vl_lite_amd.sampling import SamplingParams
    from qwen25vl_lite_amd.sampling import sampler as S
    params = [SamplingParams(temperature=1.0), SamplingParams(temperature=0.8, top_k=9, seed=5), SamplingParams(), SamplingParams(temperature=0.5, min_p=0.1),
              SamplingParams(temperature=1e-50)]
    host, more = torch.zeros(200, dtype=torch.int32), (ctypes.c_int32 * 3)()
    words, flags = S._gather(params, [[]] * 5, ["any", 2, None, 1.5, 0], 100, host, more)
    rows = host.numpy()[:60].view(S._ROW)
    assert words == 61 and list(flags) == [1, 0, 1, 0] and list(more) == [1, 1, 3]
    assert rows["seeded"].tolist() == [-1, 1, 0, -1, -1] and rows["seed"][1] == 7 and not rows["u"].any()
    assert S._gather(params, [[]] * 5, [0, 2, 0, 0, 0], 100, host)[0] == -1
    assert S._gather(params[1:3], [[]] * 2, [2, 0], 100, host, more)[0] == 25 and list(more) == [1, 0, 0]
    assert S._gather(params[1:3], [[]] * 2, ["2", 0], 100, host, more)[0] == -1


@pytest.mark.parametrize("error", ["build", "load"])
def test_sampler_without_its_native_gather(error, monkeypatch):
    """Where the interpreter's headers are missing the settings are gathered by Python's loop: tried once, refused from then on."""
    from qwen25vl_lite_amd.ops.library import KernelBuildError
    from qwen25vl_lite_amd.sampling import SamplingParams
    from qwen25vl_lite_amd.sampling import sampler as S
    tried = []

    def missing(stem, **how):
        tried.append(stem)
        raise KernelBuildError("Python.h: no such file") if error == "build" else OSError("undefined symbol")
    monkeypatch.setattr(S, "_gather_fn", None)
    monkeypatch.setattr(S, "load_library", missing)
    host = torch.zeros(40, dtype=torch.int32)
    for _ in range(3):
        assert S._gather([SamplingParams()], [[]], [0], 100, host)[0] == -1
    assert tried == ["sample_gather"]


@pytest.mark.parametrize("there", [True, False])
def test_everything_else_is_built_without_the_interpreters_headers(there, monkeypatch, tmp_path):
    from qwen25vl_lite_amd.ops import build_all
    stems = []
    monkeypatch.setattr(build_all, "python_headers", lambda: there)
    monkeypatch.setattr(build_all, "build_library", lambda stem, defines, **how: stems.append(stem) or str(tmp_path / f"{len(stems)}.so"))
    assert len(build_all.build_everything()) == len(build_all.LIBRARIES) - (not there)
    assert ("sample_gather" in stems) == there


def test_a_library_is_loaded_as_it_is_asked_for():
    """A handle whose calls let go of the interpreter's lock is not given to whoever asked for one that keeps it."""
    import ctypes

    from qwen25vl_lite_amd.ops.library import load_library
    plain, held = load_library("sample_gather"), load_library("sample_gather", loader=ctypes.PyDLL)
    assert not isinstance(plain, ctypes.PyDLL) and isinstance(held, ctypes.PyDLL)
    assert load_library("sample_gather") is plain and load_library("sample_gather", loader=ctypes.PyDLL) is held


@pytest.mark.parametrize("pairs, experts, outputs, k, gated, units, wide", [
    (3096, 8, 1376, 2048, 1, 256, 0), (3096, 8, 2048, 1376, 0, 256, 0), (2560, 8, 768, 2048, 1, 256, 0), (12384, 32, 2368, 3584, 1, 256, 1),
    (12384, 32, 3584, 2368, 0, 256, 1), (17982, 32, 1376, 2048, 1, 256, 0), (17982, 32, 2048, 1376, 0, 256, 1), (24576, 32, 1376, 2048, 1, 256, 1),
    (8191, 32, 2368, 3584, 1, 256, 0), (65536, 64, 768, 2048, 1, 256, 1), (1 << 20, 16, 4096, 4096, 1, 256, 1), (24576, 32, 1376, 2048, 1, 64, 1),
    (12798, 32, 768, 2048, 1, 256, 0), (5, 8, 64, 64, 1, 256, 0), (0, 8, 64, 64, 1, 256, 0), (4096, 8, 64, 64, 1, 0, 0)])
def test_where_experts_take_tiles_of_256_pairs(pairs, experts, outputs, k, gated, units, wide):
    """By the rounds of blocks that they come out in, which cross at other numbers of pairs for few experts than for many and for a
    gated product than for the one behind it."""
    import ctypes

    from qwen25vl_lite_amd.ops.kernels import _fn
    assert _fn("moe", "qvl_moe_wide_pairs", [ctypes.c_int] * 6)(pairs, experts, outputs, k, gated, units) == wide
