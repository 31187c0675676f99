"""Dispatch of bfloat16 products with many rows to the tiled kernel (``csrc/gemm_tile.hip``)."""

from __future__ import annotations

import ctypes
from functools import lru_cache
from typing import Optional

import torch

from .kernels import _check, _fn, _need, _ptr, _stream, compute_units

__all__ = ["MANY_ROWS", "takes_tile", "prefers_tile", "enough_gated", "tile_product", "slab_ranges", "tile_slabs", "prefers_heads", "tile_heads", "tile_swiglu",
           "tile_gated"]

_c_int, _c_ptr, _c_ll, _c_float = ctypes.c_int, ctypes.c_void_p, ctypes.c_longlong, ctypes.c_float
_STORE, _SLABS, _GROUPED, _HALVES = range(4)
PARTS = 256              # places of a row's sums of squares (TILE_PARTS in the source)
_REACH = 0xffff0000      # bytes that a tile's rows may span from its first


def _entry(name: str, argtypes):
    """A function of the library, looked up at its first call (a step of many layers makes several calls a layer and waits for the host)."""
    found = []

    def call(*args):
        if not found:
            found.append(_fn("gemm_tile", name, argtypes))
        return found[0](*args)
    return call


_blocks_of = lru_cache(maxsize=4096)(_entry("qvl_gemm_tile_blocks", [_c_int] * 4))      # (numbers of the sizes alone)
_splits_of = lru_cache(maxsize=4096)(_entry("qvl_gemm_tile_splits", [_c_int] * 4))
_tile = _entry("qvl_gemm_tile", [_c_ptr, _c_ll, _c_ptr, _c_ll, _c_ptr, _c_ll] + [_c_int] * 7 + [_c_float] * 3 + [_c_int, _c_int, _c_ptr])
_scaled = _entry("qvl_gemm_tile_scaled", [_c_ptr, _c_ll, _c_ptr, _c_ll, _c_ptr, _c_ll, _c_ptr, _c_int, _c_float] + [_c_int] * 6 + [_c_ptr])
_heads = _entry("qvl_gemm_tile_heads", [_c_ptr, _c_ll, _c_ptr, _c_ll] + [_c_ptr] * 6 + [_c_int] * 7 + [_c_ptr])


def takes_tile(x: torch.Tensor, weight: torch.Tensor, halves: bool = False) -> bool:
    """Whether the kernel takes ``x [M, K] @ weight[N, K].T``: bfloat16 rows on 16-byte boundaries, an inner size in steps
    of 32, and rows that lie within 32-bit offsets of a tile's first (``halves``: the up rows, N / 2 further on, too)."""
    if not (x.is_cuda and weight.is_cuda and x.dtype == weight.dtype == torch.bfloat16 and x.dim() == 2 and weight.dim() == 2):
        return False
    (m, k), (n, wk) = x.shape, weight.shape
    (ldx, sx), (ldw, sw) = x.stride(), weight.stride()
    return (k == wk and m > 0 and k > 0 and k % 32 == 0 and sx == 1 and sw == 1 and ldx % 8 == 0 and ldw % 8 == 0 and ldx >= k and ldw >= k
            and (x.data_ptr() | weight.data_ptr()) % 16 == 0 and (256 + (n // 2 if halves else 0)) * ldw * 2 < _REACH and 256 * ldx * 2 < _REACH)


MANY_ROWS = 64           # up to here the decode kernels and the library run


def prefers_tile(x: torch.Tensor, weight: torch.Tensor, halves: bool = False, gated: bool = False) -> bool:
    """Whether the kernel takes the product and is the faster way to it, uncut: more than ``MANY_ROWS`` rows, and tiles for
    three quarters of the compute units (2,048 x 3,584 x 3,584: 224 tiles, 54 us against the library's 66; 280 x 2,560 x
    2,048: 60 tiles, 34 against 24, the library cuts the inner size).  With a gated activation on the sums (``gated``), which
    takes the library another kernel, half of them suffice (22,016 x 2,048: 100 rows, 29 us against
    35; 200 rows, 35 against 41; 350 rows, 42 against 53; 37,888 x 3,584, 200 rows, 76 against 89)."""
    if x.shape[0] <= MANY_ROWS or not takes_tile(x, weight, halves):
        return False
    cus = compute_units(x.device)
    blocks = _blocks_of(x.shape[0], weight.shape[0], x.shape[1], cus)
    return 2 * blocks >= cus if gated or halves else 4 * blocks >= 3 * cus


def enough_gated(m: int, weight: torch.Tensor) -> bool:
    """The sizes' part of ``prefers_tile(gated=True)`` for ``m`` rows that are yet to be made."""
    n, k = weight.shape
    if m <= MANY_ROWS or k % 32:
        return False
    cus = compute_units(weight.device)
    return 2 * _blocks_of(m, n, k, cus) >= cus


def _launch(x, weight, out, ldo, mode, splits=1, relu2=0, gelu=0, alpha=1.0, limit=0.0, shift=0.0, shape=-1):
    m, k = x.shape
    _check(_tile(x.data_ptr(), x.stride(0), weight.data_ptr(), weight.stride(0), out.data_ptr(), ldo, m, weight.shape[0], k, mode, splits, relu2,
                 gelu, alpha, limit, shift, shape, compute_units(x.device), _stream()), "linear (tiles)")
    return out


def tile_product(x: torch.Tensor, weight: torch.Tensor, out_dtype: torch.dtype = torch.bfloat16,
                 out: Optional[torch.Tensor] = None, relu2: bool = False, shape: int = -1) -> torch.Tensor:
    """``x @ weight.T`` in ``out_dtype`` (``relu2``: the square of its positive part); ``shape`` names a tile (-1: by the
    kernel's estimate)."""
    _need(takes_tile(x, weight), "the tiled kernel does not take this product")
    m, n = x.shape[0], weight.shape[0]
    if out is None:
        out = torch.empty((m, n), dtype=out_dtype, device=x.device)
    _need(out.dtype == out_dtype and out_dtype in (torch.float32, torch.bfloat16) and tuple(out.shape) == (m, n)
          and out.stride(1) == 1 and out.stride(0) >= n and out.data_ptr() % 16 == 0, "out must be [M, N] of the output's dtype")
    return _launch(x, weight, out, out.stride(0), _SLABS if out_dtype == torch.float32 else _STORE, relu2=int(relu2), shape=shape)


def slab_ranges(x: torch.Tensor, weight: torch.Tensor) -> int:
    """Ranges of the inner size that :func:`tile_slabs` cuts a product into: 1 where tiles alone are faster, 0 where the kernel does
    not take the product or has few rows."""
    if x.shape[0] <= MANY_ROWS or not takes_tile(x, weight):
        return 0
    return _splits_of(x.shape[0], weight.shape[0], x.shape[1], compute_units(x.device))


def tile_slabs(x: torch.Tensor, weight: torch.Tensor, ranges: Optional[int] = None) -> Optional[torch.Tensor]:
    """Float32 slabs ``[ranges, M, N]`` over ranges of the inner size, whose sum in order is ``x @ weight.T``; None where the
    kernel does not take the product or is faster without a cut.  Cutting pays where the tiles alone leave compute units
    idle: 2,048 x 3,584 x 18,944 has 112 tiles of 256 x 256, two ranges take 204 us and one of 192 x 256 234 (the library 377).
    ``ranges``: :func:`slab_ranges` of the same, if the caller has it."""
    if ranges is None:
        ranges = slab_ranges(x, weight)
    if ranges <= 1:
        return None
    m, n = x.shape[0], weight.shape[0]
    out = torch.empty((ranges, m, n), dtype=torch.float32, device=x.device)
    return _launch(x, weight, out, n, _SLABS, splits=ranges)


def prefers_heads(x: torch.Tensor, weight: torch.Tensor, ranges: int, head_dim: int, rot_half: int, *rest: Optional[torch.Tensor]) -> bool:
    """Whether the stacked projection goes through :func:`tile_heads`: heads of 128 channels rotated whole, ``rest`` (bias, cache) on
    16-byte boundaries, and a product that is not cut along the inner size (``ranges``: :func:`slab_ranges`).

    Measured, the product (the library's, or slabs) and the rotation's kernel in brackets: 16 + 2 x 2 heads, inner size 2,048, 1,024 rows 23 us (27),
    2,048 rows 29 (37); 28 + 2 x 4 heads, 3,584, 512 rows 35 (34), 2,048 rows 67 (77), 4,096 rows 127 (151); 32 + 2 x 8 heads, 2,048, 300 rows
    23.1 (22.2); 64 + 2 x 8 heads, 8,192, 2,048 rows 282 (308).  Products that are cut stay so: in one chain of sums they would take 23 us (25, three
    slabs; 16 + 2 x 2 heads, 2,048, 512 rows), with an error of 2.7e-7 of the result against 1.5e-7."""
    return (ranges == 1 and head_dim == 128 and rot_half == 64
            and all(t is None or t.data_ptr() % 16 == 0 for t in rest))


def check_heads(m: int, n: int, nkv: int, page_size: int, bias, cs, slots, k_cache, v_cache) -> None:
    """Refuses what a projection with rotation and cache write of heads of 128 channels reads and writes beside its operands, where it does not fit."""
    _need(bias is None or (bias.dtype == torch.float32 and bias.shape == (n,) and bias.is_contiguous() and bias.is_cuda),
          "bias must be float32 [(nq + 2 nkv) 128]")
    _need(cs.is_cuda and cs.dtype == torch.float32 and cs.dim() == 3 and cs.shape[0] >= m and cs.shape[1:] == (64, 2)
          and cs.is_contiguous(), "cs must be float32 [M, 64, 2]")
    if nkv:
        _need(slots is not None and slots.is_cuda and slots.dtype == torch.int32 and slots.shape == (m,) and slots.is_contiguous(),
              "slots must be int32 [M]")
        _need(k_cache is not None and v_cache is not None and k_cache.is_cuda and v_cache.is_cuda
              and k_cache.dtype == v_cache.dtype == torch.bfloat16 and k_cache.is_contiguous() and v_cache.is_contiguous()
              and k_cache.shape[1:] == (nkv, page_size, 128) and v_cache.shape[1:] == (nkv, 128, page_size)
              and v_cache.shape[0] == k_cache.shape[0], "caches must be bfloat16 [pages, nkv, ps, 128] / [pages, nkv, 128, ps]")


def tile_heads(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor], cs: torch.Tensor, slots: Optional[torch.Tensor],
               k_cache: Optional[torch.Tensor], v_cache: Optional[torch.Tensor], num_q_heads: int, num_kv_heads: int, page_size: int,
               shape: int = -1) -> torch.Tensor:
    """The stacked query | key | value projection with bias, rotation and cache write on the float32 sums: the rotated queries
    ``[M, nq 128]`` (bfloat16); rotated keys and values are in their page slots.  ``cs``: :func:`kernels.rope_table`.  With ``num_kv_heads == 0`` the
    weight holds query rows only."""
    m, k = x.shape
    nq, nkv = int(num_q_heads), int(num_kv_heads)
    n = (nq + 2 * nkv) * 128
    _need(takes_tile(x, weight) and weight.shape[0] == n, "the tiled kernel does not take this projection")
    check_heads(m, n, nkv, page_size, bias, cs, slots, k_cache, v_cache)
    q_out = torch.empty((m, nq * 128), dtype=torch.bfloat16, device=x.device)
    _check(_heads(_ptr(x), x.stride(0), _ptr(weight), weight.stride(0), _ptr(bias), _ptr(cs), _ptr(slots if nkv else None), _ptr(q_out),
              _ptr(k_cache if nkv else None), _ptr(v_cache if nkv else None), m, k, nq, nkv, int(page_size), shape,
              compute_units(x.device), _stream()), "linear (tiles, rotation and cache write)")
    return q_out


def tile_swiglu(x: torch.Tensor, weight: torch.Tensor, act: str = "silu", shape: int = -1, taken: bool = False, scaled=None) -> torch.Tensor:
    """``act(gate) * up`` for a weight whose rows come in groups of 8 gate and 8 up rows: bfloat16 ``[M, N / 2]``.  ``taken``: :func:`takes_tile`
    has just said so.  ``scaled``: ``(squares, parts, eps)`` of rows that a product into the sum left (:func:`mid.mid_into`)."""
    _need((taken or takes_tile(x, weight)) and weight.shape[0] % 16 == 0, "the tiled kernel does not take this product")
    _need(act in ("silu", "gelu_tanh"), "the activation is silu or gelu_tanh")
    m, half = x.shape[0], weight.shape[0] // 2
    out = torch.empty((m, half), dtype=torch.bfloat16, device=x.device)
    if scaled is None:
        return _launch(x, weight, out, half, _GROUPED, gelu=int(act == "gelu_tanh"), shape=shape)
    squares, parts, eps = scaled
    _need(squares.is_cuda and squares.dtype == torch.float32 and squares.shape == (m, PARTS) and squares.is_contiguous(),
          "squares must be float32 [M, PARTS] on the GPU")
    _check(_scaled(x.data_ptr(), x.stride(0), weight.data_ptr(), weight.stride(0), out.data_ptr(), half, squares.data_ptr(), parts, eps, m,
                   weight.shape[0], x.shape[1], int(act == "gelu_tanh"), shape, compute_units(x.device), _stream()), "linear (tiles, scaled rows)")
    return out


def tile_gated(x: torch.Tensor, weight: torch.Tensor, alpha: float, limit: Optional[float], shift: float,
               shape: int = -1) -> torch.Tensor:
    """``g sigmoid(alpha g) (u + shift)`` for a weight of gate rows, then up rows: ``g`` capped at ``limit``, ``u`` clamped to
    ``[-limit, limit]`` (None: neither); bfloat16 ``[M, N / 2]``."""
    _need(takes_tile(x, weight, halves=True) and weight.shape[0] % 2 == 0, "the tiled kernel does not take this product")
    half = weight.shape[0] // 2
    out = torch.empty((x.shape[0], half), dtype=torch.bfloat16, device=x.device)
    return _launch(x, weight, out, half, _HALVES, alpha=float(alpha), limit=float(limit or 0.0), shift=float(shift), shape=shape)
