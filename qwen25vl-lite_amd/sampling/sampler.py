"""The device sampler: one token per logits row, chosen by a HIP kernel.

The reference samples on the host, one request at a time (reference
src/qwen25vl_lite/sampling.py:67-121, engine.py:802-829).  Here a step's rows are sampled
together on the GPU.  A row's uniform random number comes from the reference's per-token generator
rule (seed + number of tokens generated so far); the kernel draws it from the seed, and only rows
without a seed draw theirs here, from the global generator.
"""

from __future__ import annotations

import ctypes
from collections import defaultdict, deque
from typing import List, Optional, Sequence

import numpy as np
import torch

from ..ops.kernels import KernelError, _check, _fn, _stream
from ..ops.library import KernelBuildError, load_library
from .params import SamplingParams

__all__ = ["sample_rows", "sample_rows_begin", "sample_slots_begin", "PendingSample", "uniform_for", "uniform_from"]

_ROW = np.dtype([("temperature", "<f4"), ("top_p", "<f4"), ("min_p", "<f4"), ("u", "<f4"),
                 ("repetition", "<f4"), ("presence", "<f4"), ("frequency", "<f4"), ("top_k", "<i4"),
                 ("prev_begin", "<i4"), ("prev_end", "<i4"), ("seed", "<u4"), ("seeded", "<i4")])


def uniform_from(seed: Optional[int], step: int) -> float:
    """The uniform number in [0, 1) for output token number ``step`` of a request with this seed
    (None: from the global generator): a generator seeded with ``seed + step`` draws it
    (the rule of reference engine.py:823-829)."""
    if seed is None:
        return float(torch.rand(1).item())
    gen = torch.Generator()
    gen.manual_seed(int(seed) + int(step))
    return float(torch.rand(1, generator=gen).item())


def uniform_for(params: SamplingParams, step: int) -> float:
    """The uniform number in [0, 1) for a request's output token number ``step``."""
    return 0.0 if params.temperature <= 0 else uniform_from(params.seed, step)


def _seed_words(seeds: np.ndarray, steps: np.ndarray) -> np.ndarray:
    """What :func:`uniform_from`'s generators start from: the lower 32 bits of ``seed + step`` (int64 arrays)."""
    return (seeds.astype(np.uint64) + steps.astype(np.uint64)).astype(np.uint32)


def _int32_ids(flat: Sequence) -> np.ndarray:
    """Token ids as int32 ``[L]`` (one zero for none)."""
    try:
        ids = np.asarray(flat or [0], np.int32)
        if ids.ndim == 1:
            return ids
    except (TypeError, ValueError):
        pass
    return np.asarray([int(t) for t in flat], np.int32)   # other types than Python's and numpy's, or arrays of one id each


class _Pinned:
    """Pinned host buffers of int32, each with its event and one holder from :meth:`take` to :meth:`give`, on any thread.
    Of those given back ``KEPT`` a device stay; ``idle`` of them are left alone, so that a copy asked for lately is not waited for
    (0: buffers are given back when their copy is done)."""
    KEPT = 8

    def __init__(self, idle: int, least: int):
        self._idle, self._least, self._free = idle, least, defaultdict(deque)

    def take(self, words: int, device: torch.device):
        """A buffer of at least ``words`` that no copy uses any more: ``(host tensor, event)``."""
        free = self._free[device.index or 0]
        try:
            slot = free.popleft() if len(free) > self._idle else None
        except IndexError:          # (another thread was faster)
            slot = None
        if slot is None or slot[0].numel() < words:
            return torch.empty(max(self._least, 2 * words), dtype=torch.int32, pin_memory=True), torch.cuda.Event()
        if self._idle:
            slot[1].synchronize()       # the copy that last used this buffer is done (those given back at once have been waited for)
        return slot

    def give(self, slot, device: torch.device) -> None:
        free = self._free[device.index or 0]
        if len(free) < self.KEPT:
            free.append(slot)


_up, _down = _Pinned(3, 8192), _Pinned(0, 256)      # the rows' settings on their way to the device, sampled ids on theirs to the host


def _send(slot, words: int, device: torch.device) -> torch.Tensor:
    """The buffer's first ``words`` on the device; the buffer is given back."""
    host, copied = slot
    buf = torch.empty(words, dtype=torch.int32, device=device)
    buf.copy_(host[:words], non_blocking=True)
    copied.record()
    _up.give(slot, device)
    return buf


_ROW_WORDS = _ROW.itemsize // 4


def _gather(params, prev_ids, steps, vocab: int, host: torch.Tensor, more=None):
    """The rows' settings and ids into ``host`` by native code: ``(words, flags)``; words are -1 where a row is not of
    the usual kind, below that minus the words needed.  ``more``: three int32 that are told whether any row that draws has a cut, has none,
    and how many draw without a seed; their ``seeded`` is -1 then, where without ``more`` they are not of the usual kind."""
    global _gather_fn
    if _gather_fn is None:
        try:
            lib = load_library("sample_gather", loader=ctypes.PyDLL)
        except (KernelBuildError, OSError):      # (no headers of this interpreter, say.)  The caller's loop does the same
            _gather_fn = False
        else:
            fn = lib.qvl_sample_gather
            fn.restype = ctypes.c_long
            fn.argtypes = [ctypes.py_object] * 3 + [ctypes.c_long] * 2 + [ctypes.c_void_p, ctypes.c_long] + [ctypes.c_void_p] * 2
            _gather_fn = fn
    flags = _Flags()
    if _gather_fn is False:
        return -1, flags
    return _gather_fn(params, prev_ids, steps, len(params), vocab, host.data_ptr(), host.numel(), flags, more), flags


_gather_fn = None
_Flags, _More = ctypes.c_int32 * 4, ctypes.c_int32 * 3


class PendingSample:
    """Sampled ids that are on their way: ``device_ids`` (int32 ``[M]``, valid for kernels queued
    after the sampler on the same stream) and :meth:`result`, which waits for the host copy."""

    _slot = None

    def __init__(self, device_ids: torch.Tensor):
        m = device_ids.numel()
        self.device_ids = device_ids
        self._slot = host, event = _down.take(m, device_ids.device)
        self._host = host[:m]
        self._host.copy_(device_ids, non_blocking=True)
        event.record()

    def result(self) -> List[int]:
        slot = self._slot
        if slot is not None:
            slot[1].synchronize()
            # of several threads the first keeps its ids, and gives the buffer back only then
            self.__dict__.setdefault("_ids", self._host.tolist())
            if self.__dict__.pop("_slot", None) is not None:
                _down.give(slot, self.device_ids.device)
        return self._ids


def sample_rows(logits: torch.Tensor, params: Sequence[SamplingParams], prev_ids: Sequence[Sequence[int]],
                steps: Sequence[int], uniforms: Optional[Sequence[float]] = None) -> List[int]:
    """Sample a token for each row of float32 ``logits [M, vocab]`` on the GPU.

    ``prev_ids[m]`` are the tokens request ``m`` has generated so far (for the penalties) and
    ``steps[m]`` their number (for the seed rule).  ``uniforms`` overrides the random numbers.
    """
    return _sample_rows(logits, params, prev_ids, steps, uniforms, wait=True) or []


def sample_rows_begin(logits: torch.Tensor, params: Sequence[SamplingParams], prev_ids: Sequence[Sequence[int]],
                      steps: Sequence[int], uniforms: Optional[Sequence[float]] = None) -> Optional[PendingSample]:
    """Queue the sampling of :func:`sample_rows` and the copy of its ids to the host; nothing is
    waited for.  None for no rows."""
    return _sample_rows(logits, params, prev_ids, steps, uniforms, wait=False)


def _sample_rows(logits, params, prev_ids, steps, uniforms, wait: bool):
    if not logits.is_cuda:
        raise KernelError("sampling has no CPU path: logits must be on the GPU")
    if logits.dtype != torch.float32 or logits.dim() != 2 or not logits.is_contiguous():
        raise KernelError("logits must be contiguous float32 [M, vocab]")
    m, vocab = logits.shape
    if not (len(params) == len(prev_ids) == len(steps) == m):
        raise ValueError("one SamplingParams, token list and step per logits row is needed")
    if m == 0:
        return None
    rows = np.zeros(m, _ROW)
    flat: List[int] = []
    first = params[0]
    if (uniforms is None and first.temperature <= 0 and first.repetition_penalty == 1.0 and first.presence_penalty == 0.0
            and first.frequency_penalty == 0.0 and all(p is first or p == first for p in params)):
        # one greedy setting for the whole batch (the usual decode step): fill the rows at once
        rows[:] = (first.temperature, first.top_p, first.min_p, 0.0, 1.0, 0.0, 0.0, first.top_k if first.top_k else -1, 0, 0, 0, 0)
        return _launch(logits, rows, flat, wait)
    if uniforms is None:
        with torch.cuda.device(logits.device):
            slot, more = _up.take(m * _ROW_WORDS + 1, logits.device), _More()
            words, flags = _gather(params, prev_ids, steps, vocab, slot[0], more)
            if words < -1:
                _up.give(slot, logits.device)
                slot = _up.take(-words, logits.device)
                words, flags = _gather(params, prev_ids, steps, vocab, slot[0], more)
            if words > 0:
                if more[2]:
                    rows = slot[0].numpy()[:m * _ROW_WORDS].view(_ROW)
                    for i in np.nonzero(rows["seeded"] < 0)[0]:
                        rows["u"][i], rows["seeded"][i] = uniform_from(None, 0), 0
                return _queue(logits, _send(slot, words, logits.device), *flags, more[0], more[1], wait)
            _up.give(slot, logits.device)
    filled = []
    for i, p in enumerate(params):
        need_prev = p.repetition_penalty != 1.0 or p.presence_penalty != 0.0 or p.frequency_penalty != 0.0
        begin = len(flat)
        if need_prev:
            flat.extend(prev_ids[i])
        u, word, seeded = 0.0, 0, 0
        if uniforms is not None:
            u = uniforms[i]
        elif p.temperature > 0:
            start = None if p.seed is None else int(p.seed) + int(steps[i])
            if start is not None and -(1 << 63) <= start < 1 << 64:
                word, seeded = start & 0xffffffff, 1
            else:
                u = uniform_from(p.seed, steps[i])      # the global generator; a seed no generator takes raises
        filled.append((p.temperature, p.top_p, p.min_p, u, p.repetition_penalty, p.presence_penalty, p.frequency_penalty,
                       p.top_k if p.top_k else -1, begin, len(flat), word, seeded))
    rows[:] = filled
    return _launch(logits, rows, flat, wait)


def sample_slots_begin(logits: torch.Tensor, records, slots: Sequence[int], prev_ids: Sequence[Sequence[int]],
                       uniforms: Optional[Sequence[float]] = None) -> Optional[PendingSample]:
    """:func:`sample_rows_begin` for requests whose settings and sampler state lie in their slots
    (``records``: :class:`~qwen25vl_lite_amd.cache.slots.SlotRecords`): row ``m`` of the logits belongs to the
    request in slot ``slots[m]``.  The rows' settings are gathered by slot index; only rows with
    penalties (their generated tokens, ``prev_ids[m]``) and rows that draw without a seed are visited one by one."""
    if not logits.is_cuda:
        raise KernelError("sampling has no CPU path: logits must be on the GPU")
    if logits.dtype != torch.float32 or logits.dim() != 2 or not logits.is_contiguous():
        raise KernelError("logits must be contiguous float32 [M, vocab]")
    m = logits.shape[0]
    at = np.asarray(slots, np.int64)
    if at.shape != (m,) or len(prev_ids) != m:
        raise ValueError("one slot and token list per logits row is needed")
    if m == 0:
        return None
    rows = np.zeros(m, _ROW)
    for name in ("temperature", "top_p", "min_p", "top_k", "repetition", "presence", "frequency"):
        rows[name] = getattr(records, name)[at]
    flat: List[int] = []
    draws = rows["temperature"] > 0
    penal = (rows["repetition"] != 1.0) | (rows["presence"] != 0.0) | (rows["frequency"] != 0.0)
    for i in np.nonzero(penal)[0]:
        rows["prev_begin"][i] = len(flat)
        flat.extend(prev_ids[i])
        rows["prev_end"][i] = len(flat)
    if uniforms is not None:
        for i in np.nonzero(draws)[0]:
            rows["u"][i] = uniforms[i]
    else:
        seeds = records.seed[at]
        seeded = draws & (seeds >= 0)
        rows["seeded"] = seeded
        rows["seed"] = np.where(seeded, _seed_words(seeds, records.generated[at]), 0)
        for i in np.nonzero(draws & ~seeded)[0]:
            rows["u"][i] = uniform_from(None, 0)
    return _launch(logits, rows, flat)


_SHORT, _LONG = 1, 2      # the kernel's ways to a row's token


def _launch(logits: torch.Tensor, rows: np.ndarray, flat: List[int], wait: bool = False):
    """Send the rows' settings to the device and queue the sampler (see :func:`_queue`)."""
    vocab = logits.shape[1]
    draws = rows["temperature"] > 0
    flags = (False,) * 6
    if draws.any():
        top_k, top_p = (rows["top_k"] > 0) & (rows["top_k"] < vocab), rows["top_p"] < 1.0
        cut = top_k | top_p | (rows["min_p"] > 0)
        flags = (True, (draws & (rows["prev_end"] > rows["prev_begin"])).any(), (draws & top_k).any(), (draws & top_p).any(),
                 (draws & cut).any(), (draws & ~cut).any())
    with torch.cuda.device(logits.device):
        packed = np.concatenate([rows.view(np.int32), _int32_ids(flat)])
        slot = _up.take(packed.size, logits.device)
        slot[0].numpy()[:packed.size] = packed
        return _queue(logits, _send(slot, packed.size, logits.device), *flags, wait)


def _queue(logits: torch.Tensor, buf: torch.Tensor, draws, penalised, top_k, top_p, cut, whole, wait: bool):
    """Queue the sampler for the settings in ``buf`` (the rows, then generated ids): a :class:`PendingSample`.  With ``wait``
    the ids, and the passes for rows that the short way does not settle are queued only if there are any (a row that draws from all of its
    scores is one, which is known before).
    ``draws``, ``penalised``, ``top_k``, ``top_p``: whether any row draws, draws with generated ids, has these cuts; ``cut``, ``whole``: draws
    with a cut, with none."""
    m, vocab = logits.shape
    c_ptr, c_int = ctypes.c_void_p, ctypes.c_int
    fn = _fn("sample", "qvl_sample_rows", [c_ptr] * 7 + [c_int] * 6 + [c_ptr])
    parts_bytes = _fn("sample", "qvl_sample_parts_bytes", [c_int], restype=ctypes.c_longlong)
    dev = logits.device
    scores = scratch = None
    if draws:
        scratch_bytes = _fn("sample", "qvl_sample_scratch_bytes", [], restype=ctypes.c_longlong)
        scratch = torch.empty(m * scratch_bytes(), dtype=torch.uint8, device=dev)
        # rows that draw with penalties have their scores written out; the passes read the others' logits as they are
        if penalised:
            scores = torch.empty_like(logits)
    parts = torch.empty(m * parts_bytes(vocab), dtype=torch.uint8, device=dev)
    out = torch.empty(m + 1, dtype=torch.int32, device=dev)      # the ids, and how many rows go the long way

    def queue(ways):
        at = buf.data_ptr()
        _check(fn(logits.data_ptr(), None if scores is None else scores.data_ptr(), at, at + 4 * _ROW_WORDS * m,
                  None if scratch is None else scratch.data_ptr(), parts.data_ptr(), out.data_ptr(), m, vocab, int(top_k),
                  int(top_p), int(cut), ways, _stream()), "sample_rows")
    if not wait or scratch is None or whole:
        queue(_SHORT | _LONG)
        pending = PendingSample(out[:m])
        return pending.result() if wait else pending
    queue(_SHORT)
    ids = PendingSample(out).result()
    if ids.pop():
        queue(_LONG)
        ids = PendingSample(out[:m]).result()
    return ids
