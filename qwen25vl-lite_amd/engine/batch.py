"""Building one step's batch: from (request, its next tokens) to the flat device arrays.

A step takes any mix of prompt portions and single decoded tokens.  Each entry contributes a
contiguous run of tokens; the arrays say, per token, its id, its position rows, its request
and its index in the sequence, and per cache group where its keys and values go; per request,
where its run starts, how long its context is after the step, its pages and its state slot.
All integer arrays of a step travel to the device in one copy.
"""

from __future__ import annotations

from dataclasses import dataclass, field
from typing import List, Optional, Sequence

import numpy as np
import torch

from ..cache.manager import CacheManager
from ..parts.base import GroupStep, StepContext

__all__ = ["StepEntry", "build_step"]


@dataclass
class StepEntry:
    """A request's part in a step: ``tokens`` follow the ``start`` tokens already in the cache.

    ``positions`` gives the position rows of these tokens (``[rows][len(tokens)]``); None means
    text positions, ``start + i + rope_delta`` on every row (reference rope.py:238-247).
    ``want`` lists the places among ``tokens`` whose logits are asked for.
    """

    req_id: object
    tokens: Sequence[int]
    start: int
    want: Sequence[int] = ()
    positions: Optional[Sequence[Sequence[int]]] = None
    rope_delta: int = 0


def _align(n: int, a: int = 4) -> int:
    return (n + a - 1) // a * a


# A run's page slots are worked out by arrays from this many tokens on, one by one below (eight runs of 5 tokens 176 us of the host so, by arrays 214; one of
# 16 79 and 84, of 32 84 and 86, of 48 88 and 87, of 128 101 and 90).
ARRAY_RUN = 40


def build_step(entries: Sequence[StepEntry], cache: CacheManager, position_rows: int, dtype: torch.dtype,
               device: torch.device, vocab_size: Optional[int] = None) -> StepContext:
    """Lay out the batch (pages must have been reserved) and copy it to the device."""
    if not entries:
        raise ValueError("a step needs at least one entry")
    n_total = sum(len(e.tokens) for e in entries)
    r = len(entries)
    ngroups = len(cache.groups)
    ps = cache.page_size

    token_ids = np.empty(n_total, np.int32)
    positions = np.empty((position_rows, n_total), np.int32)
    token_req = np.empty(n_total, np.int32)
    token_seqpos = np.empty(n_total, np.int32)
    cu_q = np.zeros(r + 1, np.int32)
    ctx_len = np.empty(r, np.int32)
    req_slots = np.empty(r, np.int32)
    slot_maps = [np.empty(n_total, np.int32) for _ in range(ngroups)]
    logit_rows: List[int] = []
    seen = set()
    held = [cache.requests[e.req_id] for e in entries]
    width = max([1] + [len(t) for rp in held for t in rp.tables])
    tables = [np.full((r, width), -1, np.int32) for _ in range(ngroups)]

    at = 0
    for i, (e, rp) in enumerate(zip(entries, held)):
        n = len(e.tokens)
        if n == 0:
            raise ValueError(f"request {e.req_id!r} brings no tokens to the step")
        if e.req_id in seen:
            raise ValueError(f"request {e.req_id!r} appears twice in one step")
        seen.add(e.req_id)
        if rp.num_tokens != e.start:
            raise ValueError(f"request {e.req_id!r}: the cache holds {rp.num_tokens} tokens, "
                             f"the step continues from {e.start}")
        if n == 1 and e.positions is None and vocab_size is not None and type(e.tokens[0]) is int:
            # a decoded token beside prompt portions, one of many: a store each instead of arrays of one (24 beside a portion of 232, with the
            # portion's slots by arrays, too: 208 us of the host for 410)
            start, token = e.start, e.tokens[0]
            if not 0 <= token < vocab_size:
                raise ValueError(f"request {e.req_id!r}: token id outside [0, {vocab_size})")
            token_ids[at] = token
            token_seqpos[at] = start
            token_req[at] = i
            positions[:, at] = start + int(e.rope_delta)
            cu_q[i + 1] = at + 1
            ctx_len[i] = start + 1
            req_slots[i] = rp.slot
            for g, t in enumerate(rp.tables):
                page = t[start // ps]
                slot_maps[g][at] = page * ps + start % ps if page >= 0 else cache.slot_mapping(e.req_id, g, start, start + 1)[0]
                tables[g][i, :len(t)] = t
            for w in e.want:
                if int(w) != 0:
                    raise ValueError(f"request {e.req_id!r}: wanted place {w} is outside its 1 tokens")
                logit_rows.append(at)
            at += 1
            continue
        ids = np.asarray(e.tokens, dtype=np.int64)
        if vocab_size is not None and (ids.min() < 0 or ids.max() >= vocab_size):
            raise ValueError(f"request {e.req_id!r}: token id outside [0, {vocab_size})")
        token_ids[at:at + n] = ids
        seq = np.arange(e.start, e.start + n, dtype=np.int32)
        token_seqpos[at:at + n] = seq
        token_req[at:at + n] = i
        if e.positions is None:
            positions[:, at:at + n] = seq + np.int32(e.rope_delta)
        else:
            pos = np.asarray(e.positions, dtype=np.int64)
            if pos.shape != (position_rows, n):
                raise ValueError(f"request {e.req_id!r}: positions must be [{position_rows}, {n}], got {pos.shape}")
            positions[:, at:at + n] = pos
        cu_q[i + 1] = at + n
        ctx_len[i] = e.start + n
        req_slots[i] = rp.slot
        for g, t in enumerate(rp.tables):
            slots = None
            if n < ARRAY_RUN:
                tables[g][i, :len(t)] = t
            else:
                pages = np.asarray(t, np.int32)
                tables[g][i, :len(t)] = pages
                pages = pages[seq // ps]
                if pages.min() >= 0:
                    slots = pages * ps + seq % ps
            slot_maps[g][at:at + n] = cache.slot_mapping(e.req_id, g, e.start, e.start + n) if slots is None else slots
        for w in e.want:
            if not 0 <= int(w) < n:
                raise ValueError(f"request {e.req_id!r}: wanted place {w} is outside its {n} tokens")
            logit_rows.append(at + int(w))
        at += n

    pieces = [token_ids, positions.reshape(-1), token_req, token_seqpos, cu_q, ctx_len, req_slots,
              np.asarray(logit_rows, np.int32)]
    for g in range(ngroups):
        pieces += [slot_maps[g], tables[g].reshape(-1)]
    offsets, total = [], 0
    for p in pieces:
        offsets.append(total)
        total += _align(p.size)
    host = torch.empty(max(total, 1), dtype=torch.int32, pin_memory=(device.type == "cuda"))
    hv = host.numpy()
    for off, p in zip(offsets, pieces):
        hv[off:off + p.size] = p
    dev = host.to(device, non_blocking=True)

    def view(k: int, shape=None):
        t = dev[offsets[k]:offsets[k] + pieces[k].size]
        return t if shape is None else t.view(shape)

    groups = [GroupStep(slot_mapping=view(8 + 2 * g), block_table=view(9 + 2 * g, (r, width)), page_size=ps)
              for g in range(ngroups)]
    return StepContext(
        num_tokens=n_total, num_reqs=r,
        token_ids=view(0), positions=view(1, (position_rows, n_total)), token_req=view(2), token_seqpos=view(3),
        cu_q=view(4), ctx_len=view(5), req_slots=view(6), groups=groups, logit_rows=view(7),
        cu_q_host=cu_q.tolist(), ctx_len_host=ctx_len.tolist(), req_slots_host=req_slots.tolist(),
        max_q_len=int(np.max(cu_q[1:] - cu_q[:-1])), max_ctx_len=int(ctx_len.max()), dtype=dtype,
    )
