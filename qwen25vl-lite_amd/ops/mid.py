"""Dispatch of bfloat16 products with some hundred rows and inner sizes of a few thousand to ``csrc/gemm_mid.hip``: small tiles over all of
the inner size, added to the residual or rotated and stored in the cache."""

from __future__ import annotations

import ctypes
from typing import Optional

import torch

from . import tile
from .kernels import _check, _fn, _need, _ptr, _stream, compute_units

__all__ = ["takes_mid", "prefers_into", "leaves", "mid_into", "prefers_heads", "mid_heads"]

_c_int, _c_ptr, _c_ll = ctypes.c_int, ctypes.c_void_p, ctypes.c_longlong
_REACH = 0xffffff00
_OUTPUTS = 64            # of a block (MID_N in the source)
PARTS = 256              # places of a row's sums of squares (MID_PARTS)
# Inner sizes up to here, and one block a compute unit at most.  A projection with rotation and cache write, for the product in slabs and the rotation's
# kernel, at 65, 160, 320 and (16 + 2 x 2 heads) 400 rows: 8 + 2 x 2 heads, inner size 1,024 8.3, 8.3, 8.5 us for 11.9, 14.2, 16.6; 16 + 2 x 2, 2,048
# 12.3, 12.8, 13.5, 15.7 for 14.3, 17.9, 21.9, 22.4; 28 + 2 x 4, 2,048 12.6, 13.3 for 15.7, 19.9; 3,072 16.3, 17.6 for 16.7, 21.8; but 3,584 20.3 (100
# rows), 23.5 (200) for 19.2, 23.4.  Two rounds of blocks: 512 rows of 16 + 2 x 2, 2,048 26.1 for 24.9.
LONGEST_HEADS = 3072
# Added to the residual, with the norm behind it, for slabs and the norm that adds them, at 160, 240, 320 and 512 rows: 1,024 x 1,024 9.9, 10.2, 10.4,
# 10.7 for 11.0, 11.8, 13.5, 14.6; 2,048 x 2,048 13.9, 15.3, 15.4, 16.5 for 14.6, 15.8, 18.8, 20.3; 2,048 x 2,560 18.1, 18.8, 19.2, 19.6 for 15.8, 18.0,
# 20.7, 22.2; 2,048 x 3,072 (240, 320) 20.0, 20.7 for 18.9, 21.6; 3,584 x 3,584 (200, 256) 22.0, 24.5 for 20.3, 22.0.  The time grows with the inner
# size and hardly with the rows, that of slabs with both: from an eighth of the inner size on.
LONGEST_INTO = 2560


def _one_round(m: int, n: int, cus: int) -> bool:
    """Whether every block of 64 outputs and 64 or 80 rows has a compute unit."""
    blocks = -(-n // _OUTPUTS)
    return blocks * -(-m // 80) <= cus


def takes_mid(x: torch.Tensor, weight: torch.Tensor) -> bool:
    """Whether the kernel takes ``x [M, K] @ weight[N, K].T``: what the tiled kernel takes, within 32-bit offsets of the first row."""
    return (tile.takes_tile(x, weight) and ((weight.shape[0] - 1) * weight.stride(0) + weight.shape[1]) * 2 < _REACH
            and ((x.shape[0] - 1) * x.stride(0) + x.shape[1]) * 2 < _REACH)


def prefers_into(m: int, k: int, weight: torch.Tensor) -> bool:
    """Whether the kernel is the fastest way to add ``m`` rows' product to the sum in front of a norm."""
    return tile.MANY_ROWS < m and k <= LONGEST_INTO and 8 * m >= k and _one_round(m, weight.shape[0], compute_units(weight.device))


def leaves(n: int) -> bool:
    """Whether a row of ``n`` outputs has a place for every block's sum of squares."""
    return n <= _OUTPUTS * PARTS


def mid_into(residual: torch.Tensor, x: torch.Tensor, weight: torch.Tensor, gain: Optional[torch.Tensor] = None):
    """``residual += x @ weight.T`` (float32, in place).  With ``gain`` (float32 ``[N]``): returns ``(rows, squares, parts)``, as
    :func:`stream.stream_into`."""
    m, n = x.shape[0], weight.shape[0]
    _need(takes_mid(x, weight), "the kernel does not take this product")
    ldh, apart = residual.stride()
    _need(residual.is_cuda and residual.dtype == torch.float32 and residual.shape == (m, n) and apart == 1 and ldh >= n,
          "the residual must be float32 [M, N] on the GPU")
    rows = squares = None
    if gain is not None:
        _need(gain.is_cuda and gain.dtype == torch.float32 and gain.shape == (n,) and gain.is_contiguous() and leaves(n),
              "gain must be float32 [N] on the GPU")
        rows = torch.empty((m, n), dtype=torch.bfloat16, device=x.device)
        squares = torch.empty((m, PARTS), dtype=torch.float32, device=x.device)
    fn = _fn("gemm_mid", "qvl_gemm_mid_into", _INTO_ARGS)
    _check(fn(x.data_ptr(), x.stride(0), weight.data_ptr(), weight.stride(0), residual.data_ptr(), ldh, _ptr(gain), _ptr(rows), _ptr(squares), m, n,
              x.shape[1], compute_units(x.device), _stream()), "linear (small tiles, into the residual)")
    return None if gain is None else (rows, squares, -(-n // _OUTPUTS))


_INTO_ARGS = [_c_ptr, _c_ll, _c_ptr, _c_ll, _c_ptr, _c_ll] + [_c_ptr] * 3 + [_c_int] * 4 + [_c_ptr]
_HEADS_ARGS = [_c_ptr, _c_ll, _c_ptr, _c_ll] + [_c_ptr] * 6 + [_c_int] * 6 + [_c_ptr]


def prefers_heads(x: torch.Tensor, weight: torch.Tensor, head_dim: int, rot_half: int, *rest: Optional[torch.Tensor]) -> bool:
    """Whether the stacked projection goes through :func:`mid_heads`: heads of 128 channels rotated whole, ``rest`` (bias, cache) on 16-byte boundaries."""
    m, k = x.shape
    return (tile.MANY_ROWS < m and k <= LONGEST_HEADS and head_dim == 128 and rot_half == 64 and _one_round(m, weight.shape[0], compute_units(x.device))
            and takes_mid(x, weight) and all(t is None or t.data_ptr() % 16 == 0 for t in rest))


def mid_heads(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor], cs: torch.Tensor, slots: Optional[torch.Tensor],
              k_cache: Optional[torch.Tensor], v_cache: Optional[torch.Tensor], num_q_heads: int, num_kv_heads: int, page_size: int) -> torch.Tensor:
    """As :func:`tile.tile_heads`."""
    m, k = x.shape
    nq, nkv = int(num_q_heads), int(num_kv_heads)
    n = (nq + 2 * nkv) * 128
    _need(takes_mid(x, weight) and weight.shape[0] == n, "the kernel does not take this projection")
    tile.check_heads(m, n, nkv, page_size, bias, cs, slots, k_cache, v_cache)
    q_out = torch.empty((m, nq * 128), dtype=torch.bfloat16, device=x.device)
    fn = _fn("gemm_mid", "qvl_gemm_mid_heads", _HEADS_ARGS)
    _check(fn(x.data_ptr(), x.stride(0), weight.data_ptr(), weight.stride(0), _ptr(bias), cs.data_ptr(), _ptr(slots if nkv else None), q_out.data_ptr(),
              _ptr(k_cache if nkv else None), _ptr(v_cache if nkv else None), m, k, nq, nkv, int(page_size), compute_units(x.device), _stream()),
           "linear (small tiles, rotation and cache write)")
    return q_out
