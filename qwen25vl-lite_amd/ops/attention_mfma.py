"""Dispatch to the matrix-core attention kernel (bfloat16, head sizes in steps of 16).

The kernel is compiled per head size (``-DHD=...``) at its first use.  A step's tokens are cut
into tiles of 16 columns, a column being a (token, query head of one key/value group) pair; the
tile list depends on the batch and on the group size only and is built once per step.
"""

from __future__ import annotations

import collections
import ctypes
from typing import NamedTuple, Optional, Tuple

import numpy as np
import torch

from .kernels import _check, _fn, _need, _ptr, _stream, int32_to_device

__all__ = ["try_attention", "supports", "tiles_for", "plan_splits"]

_c_int, _c_float, _c_ptr, _c_ll = ctypes.c_int, ctypes.c_float, ctypes.c_void_p, ctypes.c_longlong
_MAX_HD = 256
# Thresholds that follow the device: counts per compute unit (measured on 256 of them); the names below
# them hold a number instead of None where a caller (a test) fixes the count itself.
TARGET_PER_CU = 2          # from this many (tile, head) pairs a compute unit on, a wave per tile fills the device
FILL_PER_CU = 1            # with fewer cooperative blocks than this, contexts are split among blocks
WIDE_WALK_BLOCKS = 80      # the kind of the kernel whose waves carry three column tiles: walks of this many 32-key blocks on average
WIDE_BLOCKS_PER_CU = 160   # ... and this many between them (41,000 on 256 units); measured with 16, 28 and 64 query heads: 43,000 blocks of 96 a walk
                           # 111 us for 116, 98,000 of 192 217 for 235, 115,000 of 128 252 for 258, 229,000 of 224 454 for 471; but 31,000 of 240
                           # 94 for 91, 13,000 of 120 65 for 52 (fewer walks, more cuts), and 33,000 and 57,000 of 64 the same within 3 per cent
GROUPS_WALK_BLOCKS = 64    # two wave groups (block_groups): walks this long on average (64 walks of 24 blocks 26 us for 24)
TARGET_BLOCKS = None
FILL_BLOCKS = None
MIN_KEYS_PER_SPLIT = 256   # keys a split has at least
SPLIT_FROM_KEYS = 768      # shorter contexts are walked by one block: merging splits (stores, a counter and loads that go
                           # through to memory) costs a decode step 2 to 2.5 us, a block's walk some 10 us per 1,000 keys (one compute unit by
                           # itself fetches its keys and values at about 40 GB/s); whole and in two splits, 8 tokens with 28 + 2 x 4 heads: 300 keys
                           # 6.3 us and 7.6, 400 6.9 and 7.6, 512 8.6 and 8.6; one token at 500 7.1 and 7.4
HALVED_KEYS = 512          # more blocks than compute units, whose contexts are no longer, run in half the waves (COOP_WAVES in the source has both sides)
MERGE_COUNTERS = 1 << 16   # (tile, kv head) pairs whose splits one launch can merge by itself
TICKET_COUNTERS = 8 * 64   # WALK_COUNTERS_AT in the source
CUT_WALKS = 1 << 13        # walks of one launch that may be cut into parts
ALONE_KEYS = 4096          # decoded tokens beside prompt portions get a launch of their own from this context on
WIDE_CT = 3
_cu_count = {}


def _compute_units(device=None) -> int:
    key = torch.device(device).index if device is not None and torch.device(device).index is not None else torch.cuda.current_device()
    if key not in _cu_count:
        _cu_count[key] = torch.cuda.get_device_properties(key).multi_processor_count
    return _cu_count[key]


def _target_blocks(device=None) -> int:
    return TARGET_BLOCKS if TARGET_BLOCKS is not None else TARGET_PER_CU * _compute_units(device)


def _fill_blocks(device=None) -> int:
    return FILL_BLOCKS if FILL_BLOCKS is not None else FILL_PER_CU * _compute_units(device)


def supports(head_dim: int, dtype: torch.dtype) -> bool:
    return dtype == torch.bfloat16 and head_dim % 16 == 0 and 16 <= head_dim <= _MAX_HD




def block_tiles(head_dim: int, wide: bool = False) -> int:
    """Column tiles of one entry of the block list (BLK_WAVES * BLK_CT in the source)."""
    return int(_fn("attention_mfma", "qvl_attn_mfma_block_tiles", [], block_defines(head_dim, wide))())


def block_defines(head_dim: int, wide: bool) -> dict:
    """The library of the kernel for many tiles: compiled per head size, and for head sizes up to 128
    in a second kind whose waves carry three column tiles instead of two.  That kind reads its operands
    from LDS once for three tiles (a third less LDS traffic and bookkeeping per product) at the price
    of longer walks and no second group of waves (where it is taken: ``WIDE_WALK_BLOCKS``)."""
    return {"HD": head_dim, "BLK_CT": WIDE_CT} if wide and head_dim <= 128 else {"HD": head_dim}


def tiles_for(cu_q, group: int, tile_ct: int = 1) -> Tuple[np.ndarray, np.ndarray]:
    """``(tile_req, tile_ct)``: for request r with q tokens, ceil(q * group / (16 * tile_ct)) entries."""
    q = np.diff(np.asarray(cu_q, dtype=np.int64))
    cols = 16 * tile_ct
    counts = (q * group + cols - 1) // cols
    req = np.repeat(np.arange(len(q), dtype=np.int32), counts)
    starts = np.cumsum(counts) - counts
    ct = (np.arange(int(counts.sum()), dtype=np.int64) - np.repeat(starts, counts)).astype(np.int32)
    return req, ct


def plan_splits(num_tiles: int, nkv: int, max_ctx: int, device=None) -> Tuple[str, int, int]:
    """``(kernel, nsplit, least keys of a split)``.  ``"tile"``: many tiles, as in prefill: a block owns
    several tiles per wave and shares the keys through LDS.  ``"coop"``: the waves of a block share a tile (few tiles, as in decode); its keys are
    split among ``nsplit`` blocks when the context is long and the blocks are few."""
    blocks = num_tiles * nkv
    if blocks >= _target_blocks(device):
        return "tile", 1, 0
    want = (_fill_blocks(device) + blocks - 1) // blocks
    nsplit = max(1, min(want, max_ctx // MIN_KEYS_PER_SPLIT)) if max_ctx >= SPLIT_FROM_KEYS else 1
    if nsplit == 1:
        return "coop", 1, 0
    # splits begin at a multiple of 32 at or below the first key a tile sees: up to 31 keys more
    per = ((max_ctx + 31 + nsplit - 1) // nsplit + 31) // 32 * 32
    nsplit = (max_ctx + 31 + per - 1) // per
    # the kernel cuts what keys a tile has evenly; where not all blocks run at once, those of shorter contexts have fewer splits instead
    # (24 tiles of 1,040 keys at most, 8 heads, captured for 2,048: two even splits 22.5 us, one of them empty 15.9)
    return "coop", nsplit, MIN_KEYS_PER_SPLIT if blocks * nsplit <= _fill_blocks(device) else per


_queues = {}
_merge_counters = {}
taken = collections.Counter()   # launches by kind of kernel (a captured launch counts once): what a measurement reports


def _counters(device: torch.device) -> torch.Tensor:
    """Per device: the counters by which the blocks of a split attention find out which of them
    finishes last and merges.  As with the work queues, a launch finds them at zero and leaves
    them at zero, and launches on one device must follow each other on one stream."""
    key = torch.device(device).index or 0
    if key not in _merge_counters:
        _merge_counters[key] = torch.zeros(MERGE_COUNTERS, dtype=torch.int32, device=device)
    return _merge_counters[key]


def _work_queue(device: torch.device):
    """Per device: the counters of the kernel for many tiles (from which workgroups take tickets for their next walk, and by which
    the parts of a cut walk find out which of them finishes last) and how many compute units there are.  A launch finds the counters at zero and leaves them at zero; launches on one
    device share them, so they must follow each other on one stream (the engine has one).  A launch
    that reports an error has them cleared."""
    key = torch.device(device).index or 0
    if key not in _queues:
        cus = torch.cuda.get_device_properties(device).multi_processor_count
        _queues[key] = (torch.zeros(TICKET_COUNTERS + CUT_WALKS, dtype=torch.int32, device=device), cus)
    return _queues[key]


class BlockPlan(NamedTuple):
    """What the kernel for many tiles does in which order (csrc/attention_mfma.hip, qvl_attn_mfma_block_plan)."""

    items: np.ndarray       # [n, 8]: request, run of column tiles, head, first and last key block, part | parts << 16, slot, counter
    grid: int               # workgroups to launch
    places: int             # of a head (or of all, where the items name their heads): workgroups that have an item to begin with
    partials: int           # partial results of all heads
    head_slots: int         # partial results and cut walks of one head (0: the items name their heads)
    head_walks: int


def plan_walks(cu_q, ctx_len, group: int, nkv: int, window: int, places: int, groups: int, defines: dict, only=None,
               cut: bool = True) -> BlockPlan:
    """The walks of a step's runs of column tiles, cut where that keeps more of ``places`` workgroups of ``groups`` wave groups busy
    (``cut``: whether any may be)."""
    cu = np.ascontiguousarray(cu_q, dtype=np.int32)
    ctx = np.ascontiguousarray(ctx_len, dtype=np.int32)
    keep = None if only is None else np.ascontiguousarray(only, dtype=np.uint8)
    cols = 16 * int(_fn("attention_mfma", "qvl_attn_mfma_block_tiles", [], defines)())
    # walks at most, and a part that is cut off fills its place or ends its walk
    room = (int(cu[-1]) * group // cols + len(ctx)) * nkv + places
    out, head = np.empty((room, 8), dtype=np.int32), np.zeros(6, dtype=np.int32)
    fn = _fn("attention_mfma", "qvl_attn_mfma_block_plan", [_c_ptr] * 3 + [_c_int] * 7 + [_c_ptr, _c_ll, _c_ptr], defines)
    _check(fn(cu.ctypes.data, ctx.ctypes.data, None if keep is None else keep.ctypes.data, len(ctx), group, nkv, window, places,
              groups, CUT_WALKS if cut else 0, out.ctypes.data, room, head.ctypes.data), "paged_attention (plan of the walks)")
    grid, count, taken_places, partials, head_slots, head_walks = (int(x) for x in head)
    return BlockPlan(out[:count], grid, taken_places, partials, head_slots, head_walks)


def _step_tiles(step, group: int, tile_ct: int, device, only=None):
    """The step's entries on the device; ``only``: a tuple of 0/1 per request, entries of the others left out."""
    cache = step.derived
    key = ("tiles", group, tile_ct, only)
    if key not in cache:
        req, ct = tiles_for(step.cu_q_host, group, tile_ct)
        if only is not None:
            keep = np.asarray(only, dtype=bool)[req]
            req, ct = req[keep], ct[keep]
        both = int32_to_device(np.concatenate([req, ct]), device)
        cache[key] = (both[:len(req)], both[len(req):], len(req))
    return cache[key]


MANY_REQUESTS = 64         # from here on a step's requests are counted by arrays


def _count_tiles(step, group: int, tile_ct: int, only=None) -> int:
    """Entries of ``tile_ct`` column tiles that the step's requests make."""
    key = ("count of tiles", group, tile_ct, only)       # the same for every layer of the step
    if key not in step.derived:
        entries = _entries(step, group, tile_ct, only)[0]
        step.derived[key] = int(entries.sum()) if isinstance(entries, np.ndarray) else sum(entries)
    return step.derived[key]


def _entries(step, group: int, tile_ct: int, only=None):
    """Per request ``(entries of tile_ct column tiles, tokens, context)``, as lists of plain integers (a step of few requests waits for
    nothing but the host, and an array of one takes 8 us for 1) or as arrays (of 200 requests both counts 29 us for 59, of 64 20 for 21)."""
    cu, ctx, cols = step.cu_q_host, step.ctx_len_host, 16 * tile_ct
    if len(ctx) >= MANY_REQUESTS:
        if ("tokens", only) not in step.derived:
            q = np.diff(np.asarray(cu, dtype=np.int64))
            step.derived["tokens", only] = (q if only is None else q * np.asarray(only, dtype=np.int64), np.asarray(ctx, dtype=np.int64))
        q, ctx = step.derived["tokens", only]
        return (q * group + cols - 1) // cols, q, ctx
    if type(cu) is not list or type(ctx) is not list:
        cu, ctx = [int(x) for x in cu], [int(x) for x in ctx]
    q = [end - begin for begin, end in zip(cu, cu[1:])]
    if only is not None:
        q = [n if keep else 0 for n, keep in zip(q, only)]
    return [(n * group + cols - 1) // cols for n in q], q, ctx


def _walk_blocks(step, group: int, tile_ct: int, only=None) -> int:
    """About how many 32-key blocks the step's entries of ``tile_ct`` column tiles walk, for one key/value head."""
    entries, q, ctx = _entries(step, group, tile_ct, only)
    if isinstance(entries, np.ndarray):
        return int((entries * np.maximum(1, (ctx - q // 2 + 31) // 32)).sum())
    return sum([e * ((c - n // 2 + 31) // 32 or 1) for e, n, c in zip(entries, q, ctx)])


def _step_walks(step, group: int, nkv: int, hd: int, window: int, device, only=None, force_wide=None, force_groups=None):
    """``(wide, wave groups, defines, plan, its items on the device)`` of the step's prompt portions, the same for every layer with
    these heads.

    A step that is captured for contexts of up to some length has walks of lengths that nobody knows yet.  They stay whole and are taken by
    tickets: cut as if all were as long as they may become, most parts would be empty (28 + 2 x 4 heads of 128, 200 decoded tokens at 275 to
    1,100 keys, captured for 2,048: 78 us, whole 57; at 450 to 1,800 116 and 103; 160 with 16 + 2 x 4 heads of 256 at 70 to 280, for 512: 42 and 33)."""
    key = ("walks", group, nkv, hd, window, only, force_wide, force_groups)
    if key in step.derived:
        return step.derived[key]
    cus = _work_queue(device)[1]
    num_tiles, blocks = _count_tiles(step, group, block_tiles(hd), only), _walk_blocks(step, group, block_tiles(hd), only)
    wide = force_wide
    if wide is None:
        # a run of twelve tiles that ends early walks for nothing more often than one of eight
        wide = (hd <= 128 and blocks >= WIDE_WALK_BLOCKS * num_tiles and blocks * nkv >= WIDE_BLOCKS_PER_CU * cus
                and _walk_blocks(step, group, block_tiles(hd, True), only) * WIDE_CT <= 1.04 * 2 * blocks)
    defines = block_defines(hd, wide)
    per_cu = int(_fn("attention_mfma", "qvl_attn_mfma_block_per_cu", [], defines)())
    known = getattr(step, "lengths_known", True)
    groups = force_groups
    if groups is None:
        groups = 1 if wide or known and blocks < GROUPS_WALK_BLOCKS * num_tiles else block_groups(num_tiles * nkv, cus * per_cu, hd, known)
    plan = plan_walks(step.cu_q_host, step.ctx_len_host, group, nkv, window, cus * (per_cu if groups == 1 else 1), groups, defines, only,
                      cut=known)
    step.derived[key] = (wide, groups, defines, plan, int32_to_device(plan.items.reshape(-1), device))
    return step.derived[key]


def long_single_tiles(step, group: int, nkv: int, device=None):
    """In a step that has prompt portions too: the requests whose tokens make one tile only
    (decoded tokens) if they are few and their contexts long, as a tuple of 0/1 per request, else
    None.  Planned together with the portions, each of them gets one workgroup (or one block) that
    walks its whole context, and that walk is what the step then waits for; in a launch of their
    own their contexts are split among blocks (measured at the 7B decoder's heads: 8 decoded tokens
    at 8,192 keys beside a portion of 256 take 87 us together, 32 and 13 apart).  Below
    ``ALONE_KEYS`` the two launches, one after the other, cost more than the walks they shorten."""
    key = ("long single tiles", group, nkv)       # the same for every layer of the step
    if key not in step.derived:
        step.derived[key] = _long_single_tiles(step, group, nkv, device)
    return step.derived[key]


def _long_single_tiles(step, group: int, nkv: int, device):
    q = np.diff(np.asarray(step.cu_q_host, dtype=np.int64))
    single = (q > 0) & (q * group <= 16)
    if not single.any() or single.all():
        return None
    longest = int(np.asarray(step.ctx_len_host, dtype=np.int64)[single].max())
    if longest < ALONE_KEYS or int(single.sum()) * nkv >= _fill_blocks(device):
        return None
    return tuple(int(x) for x in single)


def block_groups(walks: int, places: int, head_dim: int, cut: bool = True) -> int:
    """Wave groups per workgroup for a step of ``walks`` (entry, head) pairs on a device that holds
    ``places`` plain workgroups at a time.  Two groups (head sizes up to 128) halve a walk's time at
    a tenth less throughput: they pay where walks are so few that they are cut into many parts, of which one then adds up
    half as many (on 512 places, 68 walks of 124 key blocks 43 us for 50, of 247 62 for 71; 112 of 120 and 128 of 240 the same within 5
    per cent; 224 of 240 149 for 146).  Where none is cut, they pay as long as every walk has a place from the start, and the longest decides."""
    most = int(_fn("attention_mfma", "qvl_attn_mfma_block_max_groups", [], {"HD": head_dim})())
    return 2 if most >= 2 and walks * (4 if cut else 1) <= places else 1


_COOP_ARGS = [_c_ptr] * 4 + [_c_int] + [_c_ptr] * 4 + [_c_int, _c_ptr, _c_ptr] + [_c_int] * 4 + [_c_float, _c_int, _c_int, _c_ptr]
_HALVED_ARGS = [_c_ptr] * 4 + [_c_int] + [_c_ptr] * 4 + [_c_int] + [_c_ptr] * 3 + [_c_ll] + [_c_int] * 4 + [_c_float, _c_ptr]
_MERGED_ARGS = [_c_ptr] * 4 + [_c_int] + [_c_ptr] * 4 + [_c_int] + [_c_ptr] * 5 + [_c_ll] + [_c_int] * 4 + [_c_float, _c_int, _c_int, _c_ptr]


def _step_splits(step, group: int, nkv: int, device):
    """:func:`plan_splits` of all of the step's tokens, the same for every layer with these heads (and for as long as what it goes by)."""
    key = ("splits", group, nkv, TARGET_BLOCKS, FILL_BLOCKS, MIN_KEYS_PER_SPLIT, SPLIT_FROM_KEYS)
    if key not in step.derived:
        step.derived[key] = plan_splits(_count_tiles(step, group, 1), nkv, step.max_ctx_len, device)
    return step.derived[key]


def try_attention(q, k_cache, v_cache, block_table, step, num_q_heads: int, window: Optional[int],
                  scale: float, force_groups: Optional[int] = None, force_wide: Optional[bool] = None,
                  sinks: Optional[torch.Tensor] = None,
                  gate: Optional[torch.Tensor] = None) -> Optional[torch.Tensor]:
    """The attention through the matrix-core kernel, or None if it does not take this shape.  ``sinks`` (float32
    ``[heads]``): one more term ``exp(sink)`` in each query head's softmax denominator.  ``gate`` (float32 ``[N, heads]``,
    rows any distance apart): each head's output times the sigmoid of its number.
    Calls on one device must not overlap (one stream): the kernel for prompt portions keeps its
    work-queue counters in memory that all calls on the device share.
    ``force_groups``, ``force_wide`` (tests): the workgroup kind of the kernel for prompt portions and
    whether its waves carry three column tiles, else chosen by :func:`block_groups` and the number of walks."""
    pages, nkv, ps, hd = k_cache.shape
    if not supports(hd, q.dtype) or ps % 16:
        return None
    n, nq = q.shape[0], int(num_q_heads)
    _need(q.is_cuda and q.shape == (n, nq * hd) and q.is_contiguous(), "q must be contiguous [N, nq hd] on the GPU")
    _need(k_cache.dtype == v_cache.dtype == torch.bfloat16 and k_cache.is_contiguous() and v_cache.is_contiguous()
          and tuple(v_cache.shape) == (pages, nkv, hd, ps), "cache must be bfloat16 [pages, nkv, ps, hd] / [.., hd, ps]")
    _need(block_table.dtype == torch.int32 and block_table.dim() == 2 and block_table.is_contiguous()
          and block_table.shape[0] == step.num_reqs, "block_table must be int32 [R, width]")
    _need(nq % nkv == 0, "query heads must be a multiple of key/value heads")
    _need(sinks is None or (sinks.is_cuda and sinks.dtype == torch.float32 and sinks.shape == (nq,)
                            and sinks.is_contiguous()), "sinks must be float32 [nq] on the GPU")
    _need(gate is None or (gate.is_cuda and gate.dtype == torch.float32 and gate.shape == (n, nq) and gate.stride(1) == 1),
          "gate must be float32 [N, nq] on the GPU with contiguous rows")
    gate_args = (_ptr(gate), 0 if gate is None else gate.stride(0))
    out = torch.empty_like(q)
    defines = {"HD": hd}
    kind, nsplit, per = _step_splits(step, nq // nkv, nkv, q.device)

    def many_tiles(only):
        wide, groups, defines, plan, items = _step_walks(step, nq // nkv, nkv, hd, int(window or 0), q.device, only, force_wide, force_groups)
        fn = _fn("attention_mfma", "qvl_attn_mfma_block",
                 [_c_ptr] * 4 + [_c_int] + [_c_ptr] * 3 + [_c_int] * 5 + [_c_ptr, _c_ptr, _c_ptr, _c_ll] + [_c_int] * 4
                 + [_c_float, _c_ptr, _c_ptr, _c_int, _c_ptr], defines)
        counters = _work_queue(q.device)[0]
        partials = None
        if plan.partials:
            size = _fn("attention_mfma", "qvl_attn_mfma_block_part_bytes", [], defines)
            size.restype = ctypes.c_longlong
            partials = torch.empty(plan.partials * int(size()), dtype=torch.uint8, device=q.device)
        code = fn(_ptr(q), _ptr(k_cache), _ptr(v_cache), _ptr(block_table), block_table.shape[1], _ptr(step.cu_q),
                  _ptr(step.ctx_len), _ptr(items), plan.grid, len(plan.items), plan.places, plan.head_slots, plan.head_walks,
                  _ptr(out), _ptr(sinks), *gate_args, nq, nkv, ps, int(window or 0), float(scale), _ptr(partials), _ptr(counters),
                  groups, _stream())
        if code:
            # whatever a launch that went wrong did to the counters, the next one starts from zero
            counters.zero_()
        _check(code, "paged_attention (matrix cores)")
        taken[f"many tiles, {WIDE_CT if wide else 2} column tiles a wave, {groups} wave group{'s' if groups > 1 else ''}"] += 1

    def shared_tiles(only, nsplit, per):
        tile_req, tile_ct, num_tiles = _step_tiles(step, nq // nkv, 1, q.device, only=only)
        cu_q = step.cu_q
        if only is None and step.max_q_len == 1 and num_tiles == step.num_reqs == len(step.cu_q_host) - 1 == step.cu_q_host[-1]:
            # decoded tokens only: request i brings token i and has tile i, and the kernel is told so
            # instead of reading it (two dependent reads less before its first key is asked for)
            tile_req = tile_ct = cu_q = None
        scratch = None
        if nsplit > 1:
            floats = _fn("attention_mfma", "qvl_attn_mfma_scratch_floats", [_c_int] * 3, defines)
            floats.restype = ctypes.c_longlong
            scratch = torch.empty(int(floats(num_tiles, nkv, nsplit)), dtype=torch.float32, device=q.device)
        if nsplit == 1 and hd == 128 and step.max_ctx_len <= HALVED_KEYS and num_tiles * nkv > _fill_blocks(q.device):
            fn = _fn("attention_mfma", "qvl_attn_mfma_coop_halved", _HALVED_ARGS, defines)
            _check(fn(_ptr(q), _ptr(k_cache), _ptr(v_cache), _ptr(block_table), block_table.shape[1], _ptr(cu_q),
                      _ptr(step.ctx_len), _ptr(tile_req), _ptr(tile_ct), num_tiles, _ptr(out), _ptr(sinks), *gate_args, nq, nkv, ps,
                      int(window or 0), float(scale), _stream()), "paged_attention (matrix cores, shared tiles, half the waves)")
            taken["shared tiles, half the waves"] += 1
            return
        merged = nsplit > 1 and num_tiles * nkv <= MERGE_COUNTERS
        if merged or sinks is not None or gate is not None:
            # the block of each (tile, head) that finishes last merges the splits: one launch
            counters = _counters(q.device) if merged else None
            fn = _fn("attention_mfma", "qvl_attn_mfma_coop_merged", _MERGED_ARGS, defines)
            code = fn(_ptr(q), _ptr(k_cache), _ptr(v_cache), _ptr(block_table), block_table.shape[1], _ptr(cu_q),
                      _ptr(step.ctx_len), _ptr(tile_req), _ptr(tile_ct), num_tiles, _ptr(out), _ptr(scratch),
                      _ptr(counters), _ptr(sinks), *gate_args, nq, nkv, ps, int(window or 0), float(scale), nsplit, per, _stream())
            if code and merged:
                counters.zero_()
            _check(code, "paged_attention (matrix cores, shared tiles, merged)")
            taken["shared tiles, keys split among blocks, merged in the launch" if merged else "shared tiles"
                  + (", keys split among blocks, merged by a second launch" if nsplit > 1 else "")] += 1
            return
        fn = _fn("attention_mfma", "qvl_attn_mfma_coop", _COOP_ARGS, defines)
        _check(fn(_ptr(q), _ptr(k_cache), _ptr(v_cache), _ptr(block_table), block_table.shape[1], _ptr(cu_q),
                  _ptr(step.ctx_len), _ptr(tile_req), _ptr(tile_ct), num_tiles, _ptr(out), _ptr(scratch), nq, nkv, ps,
                  int(window or 0), float(scale), nsplit, per, _stream()),
               "paged_attention (matrix cores, shared tiles)")
        taken["shared tiles" + (", keys split among blocks, merged by a second launch" if nsplit > 1 else "")] += 1

    single = long_single_tiles(step, nq // nkv, nkv, q.device) if force_groups is None else None
    if single is not None:   # the few decoded tokens with long contexts by themselves, the rest planned anew
        longest = max(c for c, s in zip(step.ctx_len_host, single) if s)
        _, nsplit1, per1 = plan_splits(sum(single), nkv, longest, q.device)   # fewer blocks than fill the device: the kernel that splits
        shared_tiles(single, nsplit1, per1)
        rest = tuple(1 - s for s in single)
        kind, nsplit, per = plan_splits(_count_tiles(step, nq // nkv, 1, rest), nkv,
                                        max(c for c, s in zip(step.ctx_len_host, rest) if s), q.device)
        if kind == "tile":
            many_tiles(rest)
        else:
            shared_tiles(rest, nsplit, per)
    elif kind == "tile":
        many_tiles(None)
    else:
        shared_tiles(None, nsplit, per)
    return out
