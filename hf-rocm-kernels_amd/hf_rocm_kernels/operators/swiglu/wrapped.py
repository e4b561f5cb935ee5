from typing import Optional, Tuple

import torch
from torch import Tensor

from ...utils.dispatch import runs_now
from .binding import _swiglu


_swiglu_new = torch.ops._HFRK_C.swiglu_new.default
_swiglu_dynamic_new = torch.ops._HFRK_C.swiglu_dynamic_new.default
MAX_THREADS_PER_SM = 1024
_IO_DTYPES = (torch.bfloat16, torch.float16)


def swiglu_checks(
    gate_up_proj: Tensor,
    scale_tensor: Tensor,
    next_buffer: Tensor,
) -> None:
    """Same assertions as the reference (operators/swiglu/wrapped.py:11-29) plus the input dtype."""
    # Check shapes
    assert gate_up_proj.dim() == 2, f"Expected gate_up_proj to have 2 dims but got {gate_up_proj.dim() = } instead."
    assert gate_up_proj.size(1) % 2 == 0, f"Expected gate_up_proj an even number of columns: {gate_up_proj.shape}."
    assert next_buffer.size(0) == gate_up_proj.size(0), \
        f"Expected same number of rows: {next_buffer.shape = } but {gate_up_proj.shape = }."
    assert scale_tensor.numel() == 1, f"Expected {scale_tensor.numel() = } to be 1."
    # Check dtypes
    assert gate_up_proj.dtype in _IO_DTYPES, f"Expected {gate_up_proj.dtype = } to be torch.bfloat16 or torch.float16"
    # Check devices
    device = gate_up_proj.device
    assert device.type == "cuda", f"Expected gate_up_proj.device to be of type cuda, but got {device.type = } instead."
    assert scale_tensor.device == device, f"Expected {scale_tensor.device = } to be the same as {device = }"
    assert next_buffer.device == device, f"Expected {next_buffer.device = } to be the same as {device = }"
    # Check layouts
    assert gate_up_proj.is_contiguous(), f"Expected gate_up_proj to be contiguous but got {gate_up_proj.stride() = }"
    assert next_buffer.is_contiguous(), f"Expected residual to be contiguous but got {next_buffer.stride() = }"


def infer_num_threads(rows: int, force_scalar: bool, num_threads: int) -> int:
    """A valid explicit value is used as is; otherwise 256 threads per workgroup (the kernel is a grid-stride
    stream, so the count only sets the workgroup granularity).  The reference interpolates a table by number of
    rows instead (wrapped.py:31-47)."""
    if num_threads > 0 and num_threads <= MAX_THREADS_PER_SM:
        return num_threads
    return 256


def swiglu(
    gate_up_proj: Tensor,
    scale_tensor: Tensor,
    next_buffer: Optional[Tensor] = None,
    force_scalar: bool = False,
    num_threads: int = -1,
) -> Tensor:
    """Fused swiglu activation and conversion to fp8.  Can also zero a buffer with as many rows as the input.
    Args (reference: operators/swiglu/wrapped.py:49-84):
        - gate_up_proj: a 16-bit (bfloat16 or float16) tensor of shape (rows, 2*cols) in row-major format: gate
            in columns [0, cols), up in columns [cols, 2*cols)
        - scale_tensor: a fp32 one-item tensor to divide the result by before conversion to float8_e4m3fn
        - next_buffer: an optional 16-bit tensor of shape (rows, .) to initialise to zero
        - force_scalar: if True, use the one-element-per-thread kernel even when the 16-byte path applies
    Outputs:
        - a float8_e4m3fn tensor of shape (rows, cols) in row-major format
    """
    if next_buffer is None and not force_scalar and num_threads == -1 and runs_now(gate_up_proj):
        output = _swiglu_new(gate_up_proj, scale_tensor)  # the usual call as one native operator; None: not one of those
        if output is not None:
            return output
    if next_buffer is None:
        next_buffer = torch.empty(size=(gate_up_proj.size(0), 0), device=gate_up_proj.device, dtype=gate_up_proj.dtype)
    swiglu_checks(gate_up_proj, scale_tensor, next_buffer)
    num_threads = infer_num_threads(gate_up_proj.size(0), force_scalar, num_threads)
    swiglu_out = torch.empty(
        size=(gate_up_proj.size(0), gate_up_proj.size(1) // 2),
        dtype=torch.float8_e4m3fn,
        device=gate_up_proj.device,
    )
    _swiglu(
        gate_up_proj=gate_up_proj,
        scale_tensor=scale_tensor,
        swiglu_out=swiglu_out,
        next_buffer=next_buffer,
        force_scalar=force_scalar,
        num_threads=num_threads,
    )
    return swiglu_out


def swiglu_dynamic(
    gate_up_proj: Tensor,
    next_buffer: Optional[Tensor] = None,
) -> Tuple[Tensor, Tensor]:
    """SwiGLU with per-row dynamic quantisation to float8_e4m3fn (scale = row amax / 448).
    Returns (output fp8 (rows, cols), scales fp32 (rows,)).  cols % 8 == 0 and cols <= 32768."""
    if next_buffer is None and runs_now(gate_up_proj):
        output, scales = _swiglu_dynamic_new(gate_up_proj)
        if output is not None:
            return output, scales
    if next_buffer is None:
        next_buffer = torch.empty(size=(gate_up_proj.size(0), 0), device=gate_up_proj.device, dtype=gate_up_proj.dtype)
    swiglu_checks(gate_up_proj, torch.empty(1, dtype=torch.float32, device=gate_up_proj.device), next_buffer)
    rows, cols = gate_up_proj.size(0), gate_up_proj.size(1) // 2
    assert cols % 8 == 0 and cols <= 32768, f"Expected cols % 8 == 0 and cols <= 32768: {gate_up_proj.shape = }"
    output = torch.empty(size=(rows, cols), dtype=torch.float8_e4m3fn, device=gate_up_proj.device)
    scales = torch.empty(size=(rows,), dtype=torch.float32, device=gate_up_proj.device)
    torch.ops._HFRK_C.swiglu_dynamic(gate_up_proj, output, scales, next_buffer)
    return output, scales
