"""Matrix products of the step: ``x @ weight.T`` for ``weight`` as a Linear stores it.

float32 runs through hand-written kernels on the matrix cores' float32 instruction (true 32-bit, fixed summation order; plain
multiply-adds where strides or sizes do not suit it).
bfloat16 with up to 16 rows (a decode step) that is added to the residual, or gated behind such a sum, runs through the kernel whose waves share the inner
size (:mod:`~qwen25vl_lite_amd.ops.stream`): the sum leaves its new rows for the norm behind it (:class:`ScaledRows`), which then has no kernel.  What else
has up to 32 rows runs through the one that keeps the rows
(:mod:`~qwen25vl_lite_amd.ops.skinny`), which also folds the norm before a product, the residual add after it and the SwiGLU
activation into itself; up to 64 rows with many outputs through one that needs not keep them (:mod:`~qwen25vl_lite_amd.ops.rows`);
with more rows the tiled kernel runs (:mod:`~qwen25vl_lite_amd.ops.tile`), with the activation on its sums, or at some hundred rows of narrow models small
tiles over all of the inner size (:mod:`~qwen25vl_lite_amd.ops.mid`), which leave rows for a norm too.  Where the result
joins a sum anyway products may be cut along the inner size.  The vendor library's product, which the
reference's engine uses for its projections (reference src/qwen25vl_lite/text.py:61-66, 80-90), is left
for what neither takes or does as fast.
"""

from __future__ import annotations

from typing import Optional, Union

import torch

from . import kernels, mid, rows, skinny, stream, tile

__all__ = ["NormedRows", "ScaledRows", "NormAhead", "linear", "linear_into", "linear_stack", "linear_relu2", "gate_up_swiglu", "tune_library_products"]


class NormedRows:
    """``rmsnorm(h) * weight`` that has not been computed yet: a product that takes it may compute it
    on the way; anything else calls :meth:`materialize`."""

    def __init__(self, h: torch.Tensor, weight: torch.Tensor, eps: float, dtype: torch.dtype):
        self.h, self.weight, self.eps, self.dtype = h, weight, eps, dtype
        self.shape = h.shape

    def materialize(self) -> torch.Tensor:
        return kernels.add_rmsnorm(self.h, None, self.weight, self.eps, self.dtype)


class ScaledRows(NormedRows):
    """The same, with what the kernel that wrote ``h`` last left of it: ``rows`` (bfloat16) are ``h * weight``, and the first ``parts`` numbers of
    a row of ``squares`` add up to its sum of squares (:func:`stream.stream_into`).  Good until ``h`` changes."""

    def __init__(self, h, weight, eps, dtype, rows: torch.Tensor, squares: torch.Tensor, parts: int):
        super().__init__(h, weight, eps, dtype)
        self.rows, self.squares, self.parts = rows, squares, parts

    @property
    def scaled(self):
        return self.squares, self.parts, self.eps


class NormAhead:
    """The norm behind a product that is added to the residual, where what reads the norm takes :class:`ScaledRows`: the
    product's kernel leaves them in ``left`` if it can."""

    def __init__(self, weight: torch.Tensor, eps: float, dtype: torch.dtype):
        self.weight, self.eps, self.dtype = weight, eps, dtype
        self.left: Optional[ScaledRows] = None


def _many_rows(x: torch.Tensor, weight: torch.Tensor, bias, out_dtype, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    if rows.prefers_rows(x, weight) and (out is None or (out.dtype == torch.bfloat16 and out.stride(1) == 1 and out.stride(0) >= out.shape[1])):
        y = rows.rows_product(x, weight, out_dtype or torch.bfloat16, out)
        return y if bias is None else y + bias.to(y.dtype)
    if out is not None:
        if out.dtype == torch.bfloat16 and out.dim() == 2 and out.stride(1) == 1 and out.data_ptr() % 16 == 0 and tile.prefers_tile(x, weight):
            return tile.tile_product(x, weight, out=out)
        return torch.mm(x, weight.t(), out=out)
    if tile.prefers_tile(x, weight):
        y = tile.tile_product(x, weight, out_dtype or torch.bfloat16)
    elif out_dtype == torch.float32:
        y = torch.mm(x, weight.t(), out_dtype=torch.float32)  # float32 accumulator written out unrounded
    else:
        y = torch.nn.functional.linear(x, weight)
    if bias is not None:
        y = y + bias.to(y.dtype)
    return y


def linear(x: Union[torch.Tensor, NormedRows], weight: torch.Tensor, bias: Optional[torch.Tensor] = None,
           out_dtype: Optional[torch.dtype] = None) -> torch.Tensor:
    """``x [M, K] @ weight[N, K].T (+ bias)``.  ``out_dtype`` float32 is allowed for bfloat16
    operands (the products are accumulated in float32 either way).  ``x`` may be :class:`NormedRows`."""
    lazy = isinstance(x, NormedRows)
    m, k = x.shape
    if not weight.is_cuda:
        raise kernels.KernelError("linear has no CPU path: its tensors must be on the GPU")
    if weight.dtype == torch.bfloat16:
        # with more rows teams of blocks lose to the library, with many outputs to `rows` (see `wide`; it adds no bias)
        few = m <= skinny.ONE_BLOCK_ROWS and (bias is not None or not rows.wide(m, weight))
        if lazy and few and skinny.takes_resident(m, k, weight, norm=True):
            return skinny.resident_product(weight, h=x.h, norm_weight=x.weight, eps=x.eps, bias=bias,
                                           out_dtype=out_dtype or torch.bfloat16)
        if lazy:
            x = x.materialize()
        if x.dtype != torch.bfloat16:
            raise kernels.KernelError(f"linear: operands {x.dtype}/{weight.dtype} are not built")
        if few and skinny.takes_resident(m, k, weight) and _aligned(x):
            return skinny.resident_product(weight, x=x, bias=bias, out_dtype=out_dtype or torch.bfloat16)
        return _many_rows(x, weight, bias, out_dtype)
    if lazy:
        x = x.materialize()
    if not x.is_cuda:
        raise kernels.KernelError("linear has no CPU path: its tensors must be on the GPU")
    if x.dtype == torch.float32 and weight.dtype == torch.float32:
        return kernels.gemm_f32(x, weight, bias)
    raise kernels.KernelError(f"linear: operands {x.dtype}/{weight.dtype} are not built")


def linear_stack(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """``x[i] @ weight[i].T`` for ``x [S, M, K]`` and ``weight [S, N, K]``: ``[S, M, N]`` in the run dtype."""
    s, m, k = x.shape
    kernels._need(weight.dim() == 3 and weight.shape[0] == s and weight.shape[2] == k and weight.is_contiguous()
                  and x.stride(2) == 1 and x.dtype == weight.dtype, "x [S, M, K] and weight [S, N, K] of one dtype")
    kernels._dev(x, weight)
    out = torch.empty((s, m, weight.shape[1]), dtype=x.dtype, device=x.device)
    if weight.dtype == torch.bfloat16 and _aligned(x[0]) and x.stride(0) % 8 == 0 and skinny.takes_stack(m, k, weight):
        return skinny.stack_product(weight, x, out)      # a decode step's few rows: one launch
    for i in range(s):
        if weight.dtype == torch.float32:
            kernels.gemm_f32(x[i], weight[i], out=out[i])
        elif m <= skinny.ONE_BLOCK_ROWS and skinny.takes_resident(m, k, weight[i]) and _aligned(x[i]):
            skinny.resident_product(weight[i], x=x[i], out=out[i], out_dtype=torch.bfloat16)
        else:
            _many_rows(x[i], weight[i], None, torch.bfloat16, out=out[i])
    return out


def linear_relu2(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """``max(x @ weight.T, 0)^2`` in the run dtype: inside the product's kernel for few bfloat16 rows, else by a kernel
    behind it."""
    m, k = x.shape
    if (weight.dtype == torch.bfloat16 and weight.is_cuda and x.dtype == torch.bfloat16 and m <= skinny.ONE_BLOCK_ROWS
            and skinny.takes_resident(m, k, weight) and _aligned(x)):
        return skinny.resident_product(weight, x=x, epilogue=skinny.RELU2, out_dtype=torch.bfloat16)
    from .rownorm import squared_relu_
    if x.is_cuda and tile.prefers_tile(x, weight):
        return tile.tile_product(x, weight, relu2=True)
    z = linear(x, weight)
    return squared_relu_(z if z.is_contiguous() else z.contiguous())


def _aligned(x: torch.Tensor) -> bool:
    return x.stride(1) == 1 and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0


# Long inner sizes (``skinny.prefers_split``) are added in place where a norm waits for the rows that are left then; without one, up to here: the product
# and the norm behind it, in place and in slabs, 8 rows of 3,584 x 18,944 27.2 us and 29.1, 2,048 x 11,008 13.5 and 14.3, 4,096 x 14,336 25.0 and
# 25.0, 8,192 x 29,568 79.8 and 81.6; 16 rows 31.5 and 28.3, 15.3 and 15.4, 27.2 and 24.9, 83.3 and 78.3 (left for the norm: 28.4, 13.2, 24.1, 79.0).
IN_PLACE_ROWS = 8


def linear_into(residual: Optional[torch.Tensor], x: torch.Tensor, weight: torch.Tensor,
                ahead: Optional[NormAhead] = None, in_place: bool = False) -> Optional[torch.Tensor]:
    """``residual += x @ weight.T`` inside the product's kernel where that exists (few bfloat16
    rows): then None is returned (and the rows that the norm ``ahead`` asks for may be left in it); ``in_place``: the caller is no better off
    with slabs.  Otherwise what is to be added is returned and the caller hands
    it on to whoever adds it (the next norm's kernel): the product ``[M, N]``, or float32
    ``[slabs, M, N]`` whose slabs are added in order (the split kernel; the tiled one over ranges of the inner size)."""
    m, k = x.shape
    fast = x.is_cuda and x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16 and _aligned(x)
    if (fast and m <= stream.MOST_ROWS and residual is not None and residual.dtype == torch.float32 and residual.stride(1) == 1
            and (ahead is not None or (in_place and m <= IN_PLACE_ROWS) or not skinny.prefers_split(m, k, weight))
            and residual.shape == (m, weight.shape[0]) and residual.stride(0) >= residual.shape[1] and stream.takes_into(m, k, weight)):
        left = stream.stream_into(residual, x, weight, None if ahead is None else ahead.weight, taken=True)
        if left is not None:
            ahead.left = ScaledRows(residual, ahead.weight, ahead.eps, ahead.dtype, *left)
        return None
    if fast and skinny.prefers_split(m, k, weight):
        return skinny.split_product(weight, x)
    if (fast and m <= skinny.ONE_BLOCK_ROWS and residual is not None and skinny.takes_resident(m, k, weight)
            and residual.dtype == torch.float32 and residual.shape == (m, weight.shape[0]) and residual.stride(1) == 1):
        skinny.resident_product(weight, x=x, epilogue=skinny.RESIDUAL, out=residual)
        return None
    if (fast and in_place and residual is not None and residual.dtype == torch.float32 and mid.prefers_into(m, k, weight) and residual.stride(1) == 1
            and residual.shape == (m, weight.shape[0]) and residual.stride(0) >= residual.shape[1] and mid.takes_mid(x, weight)):
        left = mid.mid_into(residual, x, weight, ahead.weight if ahead is not None and mid.leaves(weight.shape[0]) else None)
        if left is not None:
            ahead.left = ScaledRows(residual, ahead.weight, ahead.eps, ahead.dtype, *left)
        return None
    if fast:
        slabs = tile.tile_slabs(x, weight)
        if slabs is not None:
            return slabs
    # Uncut with more rows: in bfloat16 (half the traffic of float32); the sum into the residual stays float32.
    return linear(x, weight, out_dtype=torch.float32 if m <= skinny.ONE_BLOCK_ROWS else None)


def tune_library_products(enable: bool = True, max_ms: int = 3000) -> None:
    """Let PyTorch's TunableOp pick the fastest library kernel for every product shape it meets
    (each new shape costs a few seconds once; its choices are kept in a per-user file under the
    temporary directory).  Meant for runs with few distinct shapes, such as a benchmark; off by
    default."""
    import os
    import tempfile

    import torch.cuda.tunable as tunable

    if enable:
        tunable.set_filename(os.path.join(tempfile.gettempdir(), f"qwen25vl_lite_amd-tunableop-{os.getuid()}.csv"))
        tunable.set_max_tuning_duration(int(max_ms))
    tunable.enable(enable)
    tunable.tuning_enable(enable)


def gate_up_swiglu(x: Union[torch.Tensor, NormedRows], weight: torch.Tensor, grouped: bool, act: str = "silu") -> torch.Tensor:
    """``act(x Wg^T) * (x Wu^T)`` (``act`` ``"silu"`` or ``"gelu_tanh"``) for ``weight`` holding gate and up rows: plain (gate rows, then up
    rows) or ``grouped`` (alternating groups of 8 gate rows and 8 up rows).  With few bfloat16 rows
    and grouped rows the activation is applied inside the product's kernel."""
    m, k = x.shape
    if grouped and isinstance(x, ScaledRows) and stream.takes_gated(m, k, weight):
        return stream.stream_gated(x.rows, weight, act, x.scaled)
    if grouped and isinstance(x, ScaledRows) and tile.MANY_ROWS < m and tile.prefers_tile(x.rows, weight, gated=True):
        return tile.tile_swiglu(x.rows, weight, act, taken=True, scaled=x.scaled)
    if (grouped and weight.dtype == torch.bfloat16 and weight.is_cuda and weight.shape[0] % 16 == 0
            and m <= skinny.ONE_BLOCK_ROWS and not rows.wide(m, weight)):
        lazy = isinstance(x, NormedRows)
        if lazy and skinny.takes_resident(m, k, weight, norm=True):
            return skinny.resident_product(weight, h=x.h, norm_weight=x.weight, eps=x.eps, epilogue=skinny.GATED[act])
        if not lazy and x.dtype == torch.bfloat16 and skinny.takes_resident(m, k, weight) and _aligned(x):
            return skinny.resident_product(weight, x=x, epilogue=skinny.GATED[act])
    if grouped and weight.shape[0] % 16 == 0:
        if isinstance(x, NormedRows):
            x = x.materialize()
        if rows.prefers_rows(x, weight):
            return rows.rows_swiglu(x, weight, act)
        if x.is_cuda and tile.prefers_tile(x, weight, gated=True):
            return tile.tile_swiglu(x, weight, act, taken=True)
    return kernels.swiglu(linear(x, weight), grouped=grouped, act=act)
