"""Dispatch of bfloat16 products with up to 64 rows and many outputs to ``csrc/gemm_rows.hip``, whose blocks need not keep the
rows."""

from __future__ import annotations

import ctypes
from typing import Optional

import torch

from . import skinny
from .kernels import _check, _fn, _need, _ptr, _stream, compute_units

__all__ = ["takes_rows", "prefers_rows", "rows_product", "rows_swiglu", "many_outputs", "rows_gated"]

_c_int, _c_ptr, _c_ll, _c_float = ctypes.c_int, ctypes.c_void_p, ctypes.c_longlong, ctypes.c_float
_REACH = 0xffffff00
MOST_ROWS = 64


def _aligned(t: torch.Tensor) -> bool:
    return t.stride(1) == 1 and t.stride(0) % 8 == 0 and t.stride(0) >= t.shape[1] and t.data_ptr() % 16 == 0


def takes_rows(x: torch.Tensor, weight: torch.Tensor) -> bool:
    """Whether the kernel takes ``x [M, K] @ weight[N, K].T``: up to 64 bfloat16 rows on 16-byte boundaries, an inner size in
    steps of 8, operands within 32-bit byte offsets."""
    return (x.dim() == 2 and x.shape[0] <= MOST_ROWS and x.is_cuda and weight.is_cuda and x.dtype == weight.dtype == torch.bfloat16 and weight.dim() == 2
            and x.shape[1] == weight.shape[1] and 0 < x.shape[0] <= MOST_ROWS and x.shape[1] > 0 and x.shape[1] % 8 == 0
            and _aligned(x) and _aligned(weight) and ((weight.shape[0] - 1) * weight.stride(0) + x.shape[1]) * 2 < _REACH
            and ((x.shape[0] - 1) * x.stride(0) + x.shape[1]) * 2 < _REACH)


def many_outputs(weight: torch.Tensor) -> bool:
    """At least 8 for each of a device's waves, eight a compute unit (10,240 x 8,192 at 19 rows 60 us, the library, which
    cuts the inner size, 41)."""
    return weight.shape[0] >= 64 * compute_units(weight.device)


def wide(m: int, weight: torch.Tensor) -> bool:
    """Whether the kernel is the fastest way to ``m`` rows: many outputs, and an inner size beyond the resident kernel's
    narrow build (a norm formed in each of its blocks takes longer than a kernel of its own), or more rows than that
    carries in one column tile.  Against
    the resident kernel at 32 rows: 22,016 x 2,048 gated 18 us for 24, with the norm in front 21 for 29; 37,888 x 3,584 45
    for 53, 49 for 64; 152,064 x 3,584 187 for 197; with 9 rows and the norm
    37,888 x 3,584 46.6 us for 50.7, with 16 47.1 for 53.9 (22,016 x 2,048 22.6 for 22.0, 23.0 for 23.5); with 1 row 48.7 for 49.7 (23.6 for
    20.9).  Against the library at 64 rows: 37,888 x 3,584 gated 51 us for 65 with the
    activation's kernel, 59,136 x 8,192 143 for 195; heads of 152,064 x 3,584 198 for 218, x 8,192 421 for 493."""
    k = weight.shape[1]
    return (m <= MOST_ROWS and many_outputs(weight)
            and (k > skinny.NARROW_K or m > skinny.ONE_TILE_ROWS or not skinny.takes_resident(m, k, weight)))


def prefers_rows(x: torch.Tensor, weight: torch.Tensor) -> bool:
    return takes_rows(x, weight) and wide(x.shape[0], weight)


def _launch(x, weight, out, mode, gelu=0, alpha=1.0, limit=0.0, shift=0.0):
    fn = _fn("gemm_rows", "qvl_gemm_rows", [_c_ptr, _c_ll, _c_ptr, _c_ll, _c_ptr, _c_ll] + [_c_int] * 5
             + [_c_float] * 3 + [_c_int, _c_ptr])
    _check(fn(_ptr(x), x.stride(0), _ptr(weight), weight.stride(0), _ptr(out), out.stride(0), x.shape[0], weight.shape[0],
              x.shape[1], mode, gelu, alpha, limit, shift, compute_units(x.device), _stream()), "linear (few rows)")
    return out


def rows_product(x: torch.Tensor, weight: torch.Tensor, out_dtype: torch.dtype = torch.bfloat16,
                 out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``x @ weight.T`` in ``out_dtype``."""
    _need(takes_rows(x, weight), "the kernel does not take this product")
    m, n = x.shape[0], weight.shape[0]
    if out is None:
        out = torch.empty((m, n), dtype=out_dtype, device=x.device)
    _need(out.dtype == out_dtype and out_dtype in (torch.float32, torch.bfloat16) and tuple(out.shape) == (m, n)
          and out.stride(1) == 1 and out.stride(0) >= n, "out must be [M, N] of the output's dtype")
    return _launch(x, weight, out, int(out_dtype == torch.float32))


def rows_swiglu(x: torch.Tensor, weight: torch.Tensor, act: str = "silu") -> torch.Tensor:
    """``act(gate) * up`` for a weight whose rows come in groups of 8 gate and 8 up rows: bfloat16 ``[M, N / 2]``."""
    _need(takes_rows(x, weight) and weight.shape[0] % 16 == 0, "the kernel does not take this product")
    _need(act in ("silu", "gelu_tanh"), "the activation is silu or gelu_tanh")
    out = torch.empty((x.shape[0], weight.shape[0] // 2), dtype=torch.bfloat16, device=x.device)
    return _launch(x, weight, out, 2, int(act == "gelu_tanh"))


def rows_gated(x: torch.Tensor, weight: torch.Tensor, alpha: float, limit: Optional[float], shift: float) -> torch.Tensor:
    """``g sigmoid(alpha g) (u + shift)`` for a weight of gate rows, then up rows: ``g`` capped at ``limit``, ``u`` clamped to
    ``[-limit, limit]`` (None: neither); bfloat16 ``[M, N / 2]``."""
    _need(takes_rows(x, weight) and weight.shape[0] % 2 == 0, "the kernel does not take this product")
    out = torch.empty((x.shape[0], weight.shape[0] // 2), dtype=torch.bfloat16, device=x.device)
    return _launch(x, weight, out, 3, alpha=float(alpha), limit=float(limit or 0.0), shift=float(shift))
