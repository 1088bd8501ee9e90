"""Linear layers of few rows on MFMA tiles (no reference counterpart: the
reference runs ``F.linear`` for every projection, tinyvllm/layers.py:80-125)."""
from __future__ import annotations

import torch

from tinyvllm.kernels._extension import (
    check, dtype_code, load_kernels, require_gpu, stream_of, values_only,
)

MAX_ROWS = 64
HALVES = (torch.bfloat16, torch.float16)


def fits(x: torch.Tensor, weight: torch.Tensor) -> bool:
    """Whether ``few_rows_linear`` takes these tensors: 1 to 64 half-precision
    rows on the GPU in 16-byte units, widths in multiples of 32, outside
    autocast and wherever more than values is asked for (autograd, forward
    mode, transforms, tracing), which only the torch ops serve."""
    if not x.is_cuda or not values_only(x, weight):
        return False
    rows, stride = x.shape, x.stride()
    columns, width = weight.shape
    return (len(rows) == 2 and 0 < rows[0] <= MAX_ROWS and x.dtype in HALVES
            and x.dtype == weight.dtype and x.get_device() == weight.get_device()
            and stride[1] == 1 and stride[0] % 8 == 0 and weight.is_contiguous()
            and columns % 32 == 0 and width % 32 == 0
            and x.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0
            and not torch.is_autocast_enabled("cuda"))


def few_rows_linear(x: torch.Tensor, weight: torch.Tensor, *, slices: int = 0,
                    silu: bool = False) -> torch.Tensor:
    """``x @ weight.T`` for up to 64 rows, accumulated in fp32.

    ``slices`` > 0 returns the fp32 partial products [slices, rows, columns]
    over that many slices of the reduction axis instead of the rounded result;
    ``silu`` takes ``weight`` as packed [gate | up] rows and returns
    ``silu(gate) * up`` [rows, columns / 2] with the rounding points of
    ``silu_and_mul`` over the rounded projection."""
    device = require_gpu(x, weight)
    if x.dim() != 2 or weight.dim() != 2 or x.shape[1] != weight.shape[1]:
        raise RuntimeError("few_rows_linear takes [rows, width] and [columns, width]")
    if x.dtype != weight.dtype or x.stride(1) != 1 or not weight.is_contiguous():
        raise RuntimeError("few_rows_linear needs one dtype, unit last stride and a "
                           "contiguous weight")
    rows, (columns, width) = x.shape[0], weight.shape
    if slices:
        out = torch.empty((slices, rows, columns), dtype=torch.float32, device=device)
    else:
        out = torch.empty((rows, columns // 2 if silu else columns), dtype=x.dtype,
                          device=device)
    check(load_kernels().tvllm_few_rows_linear(
        x.data_ptr(), x.stride(0), weight.data_ptr(), rows, columns, width, out.data_ptr(),
        slices, int(silu), dtype_code(x.dtype), stream_of(device)))
    return out
