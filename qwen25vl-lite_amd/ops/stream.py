"""Dispatch of bfloat16 products with up to 16 rows to ``csrc/gemm_stream.hip``: those that are added to the residual, and gated
ones whose rows are still to be normed.

Between two products of a decode step stands a norm.  The product that ends a sublayer adds into the float32 sum; a norm's row is the
sum's row times the norm's gain, divided by one number, the row's root mean square.  So the first product leaves the new rows times the gain, in
bfloat16, and its blocks' sums of squares (:class:`ScaledRows`), and the product behind the norm multiplies those rows and divides its sums by
the root mean square: the norm's own kernel falls away.
"""

from __future__ import annotations

import ctypes
from typing import Optional

import torch

from .kernels import _check, _fn, _need, _ptr, _stream, compute_units

__all__ = ["takes_into", "stream_into", "takes_gated", "stream_gated", "MOST_ROWS", "PARTS"]

_c_int, _c_ptr, _c_ll, _c_float = ctypes.c_int, ctypes.c_void_p, ctypes.c_longlong, ctypes.c_float
_REACH = 0xffffff00
MOST_ROWS = 16
PARTS = 256            # places of a row's sums of squares (STREAM_PARTS in the source)
MOST_TILES = 4         # tiles of 16 rows of W a block takes where the product is added to the residual (STREAM_MOST_INTO)
MOST_GATED_TILES = 16  # tiles of 8 channels (STREAM_MOST_GATED)


def _fits(m: int, k: int, weight: torch.Tensor) -> bool:
    if not (0 < m <= MOST_ROWS and k > 0 and k % 8 == 0 and weight.dtype == torch.bfloat16 and weight.dim() == 2 and weight.is_cuda):
        return False
    (n, width), (ld, apart) = weight.shape, weight.stride()
    return width == k and apart == 1 and ld % 8 == 0 and ld >= k and ((n - 1) * ld + k) * 2 < _REACH and weight.data_ptr() % 16 == 0


def _blocks(n: int, cus: int) -> int:
    return min(n, cus, PARTS)


def takes_into(m: int, k: int, weight: torch.Tensor) -> bool:
    """Whether :func:`stream_into` takes ``m`` rows of width ``k``: up to 16, an inner size in steps of 8, up to 64 outputs a compute unit."""
    n = weight.shape[0]
    return _fits(m, k, weight) and n > 0 and -(-n // _blocks(n, compute_units(weight.device))) <= 16 * MOST_TILES


def takes_gated(m: int, k: int, weight: torch.Tensor) -> bool:
    """Whether :func:`stream_gated` takes ``m`` rows of width ``k``: up to 16, up to 128 channels a compute unit."""
    n = weight.shape[0]
    if not (_fits(m, k, weight) and n > 0 and n % 16 == 0):
        return False
    blocks = min(n // 2, compute_units(weight.device))
    return -(-(-(-(n // 2) // blocks)) // 8) <= MOST_GATED_TILES


def _check_x(x: torch.Tensor, taken: bool):
    """``(m, k, rows' distance)`` of an operand that a kernel takes."""
    (m, k), (ld, apart) = x.shape, x.stride()
    _need(taken and x.is_cuda and x.dtype == torch.bfloat16 and apart == 1 and ld % 8 == 0 and ld >= k and ((m - 1) * ld + k) * 2 < _REACH
          and x.data_ptr() % 16 == 0, "the kernel does not take this product")
    return m, k, ld


_INTO_ARGS = [_c_ptr, _c_ll, _c_ptr, _c_ll, _c_ptr, _c_ll] + [_c_ptr] * 3 + [_c_int] * 4 + [_c_ptr]
_GATED_ARGS = [_c_ptr, _c_ll, _c_ptr, _c_ll, _c_ptr, _c_ll, _c_ptr, _c_int, _c_float] + [_c_int] * 5 + [_c_ptr]


def stream_into(residual: torch.Tensor, x: torch.Tensor, weight: torch.Tensor, gain: Optional[torch.Tensor] = None, taken: bool = False):
    """``residual += x @ weight.T`` (float32, in place).  ``taken``: :func:`takes_into` has just said so.  With ``gain`` (float32 ``[N]``): returns ``(rows, squares, parts)``, the new
    residual times the gain in bfloat16 and float32 ``[M, PARTS]`` whose first ``parts`` numbers of a row add up to the residual row's sum of squares."""
    m, k, ldx = _check_x(x, taken or takes_into(x.shape[0], x.shape[1], weight))
    n, (ldh, apart) = weight.shape[0], residual.stride()
    _need(residual.is_cuda and residual.dtype == torch.float32 and residual.shape == (m, n) and apart == 1 and ldh >= n,
          "the residual must be float32 [M, N] on the GPU")
    rows = squares = None
    cus = compute_units(x.device)
    if gain is not None:
        _need(gain.is_cuda and gain.dtype == torch.float32 and gain.shape == (n,) and gain.is_contiguous(), "gain must be float32 [N] on the GPU")
        rows = torch.empty((m, n), dtype=torch.bfloat16, device=x.device)
        squares = torch.empty((m, PARTS), dtype=torch.float32, device=x.device)
    fn = _fn("gemm_stream", "qvl_gemm_stream_into", _INTO_ARGS)
    _check(fn(x.data_ptr(), ldx, weight.data_ptr(), weight.stride(0), residual.data_ptr(), ldh, _ptr(gain), _ptr(rows),
              _ptr(squares), m, n, k, cus, _stream()), "linear (stream, into the residual)")
    return None if gain is None else (rows, squares, _blocks(n, cus))


def stream_gated(x: torch.Tensor, weight: torch.Tensor, act: str = "silu", scaled=None) -> torch.Tensor:
    """``act(gate) * up`` for a weight whose rows come in groups of 8 gate and 8 up rows: bfloat16 ``[M, N / 2]``.  ``scaled``: ``(squares, parts,
    eps)`` of rows that :func:`stream_into` left."""
    _need(act in ("silu", "gelu_tanh"), "the activation is silu or gelu_tanh")
    m, k, ldx = _check_x(x, takes_gated(x.shape[0], x.shape[1], weight))
    n = weight.shape[0]
    out = torch.empty((m, n // 2), dtype=torch.bfloat16, device=x.device)
    squares, parts, eps = scaled if scaled is not None else (None, 0, 0.0)
    _need(squares is None or (squares.is_cuda and squares.dtype == torch.float32 and squares.shape == (m, PARTS) and squares.is_contiguous()),
          "squares must be float32 [M, PARTS] on the GPU")
    fn = _fn("gemm_stream", "qvl_gemm_stream_gated", _GATED_ARGS)
    _check(fn(x.data_ptr(), ldx, weight.data_ptr(), weight.stride(0), out.data_ptr(), n // 2, _ptr(squares), parts, eps, m, n, k, int(act == "gelu_tanh"), compute_units(x.device), _stream()), "linear (stream, gated)")
    return out
