from typing import Optional, Tuple

import torch
from torch import Tensor

from hf_rocm_kernels import residual_rms, skinny_gemm, skinny_gemm_add, skinny_gemm_rms, skinny_gemm_scaled, skinny_gemm_swiglu, swiglu

from .. import _capi
from ..utils.dispatch import runs_now
from ..utils.weight_format import PackedWeight

_llama_mlp = torch.ops._HFRK_C.llama_mlp.default


def _native_block(attn_output, residual, residual_out, attn_copy, output, rms_weight, rms_epsilon, gate_up_weight, gate_up_input_scale,
                  gate_up_output_scale, down_weight, down_input_scale, down_output_scale, add_residual, memory=None) -> bool:
    """The fused block as one native operator, into the given tensors; False, with nothing written, if this is not one of its calls.
    For calls that run now (utils/dispatch.py).  memory: bytes of `_block_memory`; without them scratch is allocated and partial sums go to the
    stream's workspace."""
    gate_up_packed, down_packed = isinstance(gate_up_weight, PackedWeight), isinstance(down_weight, PackedWeight)
    return _llama_mlp(attn_output, residual, residual_out, attn_copy, rms_weight, rms_epsilon,
                      gate_up_weight.data if gate_up_packed else gate_up_weight, gate_up_weight.n if gate_up_packed else -1,
                      gate_up_input_scale, gate_up_output_scale, down_weight.data if down_packed else down_weight,
                      down_weight.n if down_packed else -1, down_input_scale, down_output_scale, add_residual, output, memory)


def _block_memory(rows, hidden, gate_up_weight, down_weight, device) -> Tensor:
    """Scratch and workspace of a block's calls, the workspace's arrival counters clear."""
    lib, inter = _capi.load(), down_weight.size(0)
    size = lib.hfrk_llama_mlp_scratch_bytes(rows, hidden, inter)
    size += lib.hfrk_llama_mlp_workspace_bytes(rows, hidden, inter, isinstance(gate_up_weight, PackedWeight), isinstance(down_weight, PackedWeight))
    return torch.zeros(size, dtype=torch.uint8, device=device)


def llama_mlp_combined_ops(
    attn_output: Tensor,
    residual: Tensor,
    rms_weight: Tensor,
    rms_epsilon: float,
    gate_up_weight: Tensor,
    gate_up_input_scale: Tensor,
    gate_up_output_scale: Tensor,
    down_weight: Tensor,
    down_input_scale: Tensor,
    down_output_scale: Tensor,
    gate_up_gemm_hp: Tuple[Optional[int], Optional[int]] = (None, None),
    down_gemm_hp: Tuple[Optional[int], Optional[int]] = (None, None),
    add_residual: bool = False,
    fused: bool = False,
    rms_prologue: bool = False,
) -> Tuple[Tensor, Tensor]:
    """Decoder MLP sub-block as four launches on one stream (reference: combined_ops/llama_mlp.py:7-60):
    residual RMSNorm -> fp8, gate_up GEMM, SwiGLU -> fp8, down GEMM.

    - attn_output, residual: (m, hidden) 16-bit; residual <- attn_output + residual in place
    - gate_up_weight: (hidden, 2*inter) fp8, col-major; down_weight: (inter, hidden) fp8, col-major
    - *_input_scale: the activation quantisation scale of each GEMM; *_output_scale: activation scale x weight scale
    - gate_up_gemm_hp / down_gemm_hp: accepted for signature compatibility; the library plans each GEMM itself
      (the reference forwards them as split_k / b_lanes keywords its skinny_gemm does not take)
    - add_residual: the down projection accumulates onto a copy of the updated residual instead of zeros, so
      the first output is the block's output hidden state (residual + mlp) rounded once

    - fused: three launches instead of four (plus a copy): the SwiGLU runs as the epilogue of the gate_up GEMM,
      nothing is zeroed beforehand (the GEMMs overwrite), and with add_residual the down projection reads the
      residual as its addend instead of accumulating onto a copy.  Same arithmetic, same roundings.

    - rms_prologue (with fused): two launches where the library has the prologue (up to 8 rows, hidden 4096 or 8192,
      row-major gate_up weight): the RMSNorm runs inside the gate_up GEMM, in every workgroup.  Same bits as the three
      launches, but the summed residual is returned as a new tensor and `residual` is left as it was (every workgroup of
      the fused launch reads the old residual, so it cannot be updated in place).

    RMSNorm and SwiGLU zero the buffer the following GEMM accumulates into, as in the reference.
    Returns (mlp_output, residual)."""
    del gate_up_gemm_hp, down_gemm_hp
    if fused and rms_prologue:
        swiglu_out, residual = skinny_gemm_rms(attn_output, residual, rms_weight, rms_epsilon, gate_up_input_scale, gate_up_weight,
                                               gate_up_output_scale, None, None, out_scale=down_input_scale)
        if add_residual:
            mlp_output = skinny_gemm_add(swiglu_out, down_weight, down_output_scale, None, base=residual)
        else:
            mlp_output = torch.empty(size=(attn_output.size(0), down_weight.size(1)), dtype=attn_output.dtype,
                                     device=attn_output.device)
            skinny_gemm_scaled(swiglu_out, down_weight, down_output_scale,
                               torch.ones(1, device=attn_output.device), output=mlp_output)
        return mlp_output, residual
    if fused:
        if runs_now(attn_output) and attn_output.dim() == 2:
            mlp_output = torch.empty_like(attn_output)
            if _native_block(attn_output, residual, residual, None, mlp_output, rms_weight, rms_epsilon, gate_up_weight, gate_up_input_scale,
                             gate_up_output_scale, down_weight, down_input_scale, down_output_scale, add_residual):
                return mlp_output, residual
        normalized, residual = residual_rms(input=attn_output, residual=residual, weight=rms_weight, epsilon=rms_epsilon,
                                            scale_tensor=gate_up_input_scale)
        swiglu_out = skinny_gemm_swiglu(normalized, gate_up_weight, gate_up_output_scale, None, down_input_scale,
                                        intermediate_dtype=attn_output.dtype)
        if add_residual:
            mlp_output = skinny_gemm_add(swiglu_out, down_weight, down_output_scale, None, base=residual)
        else:
            mlp_output = torch.empty(size=(attn_output.size(0), down_weight.size(1)), dtype=attn_output.dtype,
                                     device=attn_output.device)
            skinny_gemm_scaled(swiglu_out, down_weight, down_output_scale,
                               torch.ones(1, device=attn_output.device), output=mlp_output)
        return mlp_output, residual
    m = attn_output.size(0)
    dtype = attn_output.dtype

    # RMS norm (zeroes the gate_up GEMM's accumulator)
    gate_up_proj = torch.empty(size=(m, gate_up_weight.size(1)), dtype=dtype, device=attn_output.device)
    normalized, residual = residual_rms(
        input=attn_output,
        residual=residual,
        weight=rms_weight,
        epsilon=rms_epsilon,
        scale_tensor=gate_up_input_scale,
        next_buffer=gate_up_proj,
    )

    # Gate + up projection
    skinny_gemm(skinny_a=normalized, b=gate_up_weight, scale_tensor=gate_up_output_scale, output=gate_up_proj)

    # Swiglu (zeroes the down GEMM's accumulator unless it starts from the residual)
    if add_residual:
        mlp_output = residual.clone()
        swiglu_out = swiglu(gate_up_proj=gate_up_proj, scale_tensor=down_input_scale)
    else:
        mlp_output = torch.empty(size=(m, down_weight.size(1)), dtype=dtype, device=attn_output.device)
        swiglu_out = swiglu(gate_up_proj=gate_up_proj, scale_tensor=down_input_scale, next_buffer=mlp_output)

    # Down projection
    skinny_gemm(skinny_a=swiglu_out, b=down_weight, scale_tensor=down_output_scale, output=mlp_output)
    return mlp_output, residual


class LlamaMlpGraph:
    """The decoder MLP sub-block for a fixed number of rows: captured once into a HIP graph (`graph`; the reference times its kernels
    inside graphs, operators/skinny_gemm/benchmarking_fn.py:62-92, but ships no captured block), and callable.

    The graph reads `attn_output` and `residual` from buffers owned by this object: write the step's inputs with `copy_`, replay, and read the
    results from `mlp_output` / `residual`, which every replay overwrites.  A call leaves the same in the same buffers.  The usual call
    does not replay: it launches the native block on the inputs where they are, which is faster than the graph but costs about 15 us of
    host, and takes no memory and no workspace of the stream it is made on (the object owns both).  A call during a caller's capture
    is refused; `llama_mlp_combined_ops` can be captured.  Calls and replays of one object share its buffers: one at a time.
    Weights and scales are the tensors given here; replace their contents in place if they change.  Capturing needs the library's
    workspace to exist, so one eager run happens first."""

    def __init__(self, rows: int, hidden: int, rms_weight: Tensor, rms_epsilon: float, gate_up_weight, gate_up_input_scale: Tensor,
                 gate_up_output_scale: Tensor, down_weight, down_input_scale: Tensor, down_output_scale: Tensor,
                 dtype: torch.dtype = torch.bfloat16, add_residual: bool = True, fused: bool = True):
        device = rms_weight.device
        self.attn_output = torch.zeros((rows, hidden), dtype=dtype, device=device)
        self.residual = torch.zeros((rows, hidden), dtype=dtype, device=device)
        args = (rms_weight, rms_epsilon, gate_up_weight, gate_up_input_scale, gate_up_output_scale, down_weight,
                down_input_scale, down_output_scale)
        kwargs = dict(add_residual=add_residual, fused=fused)
        self._operands = args  # the captured launches read their addresses: they live as long as the graph
        self._add_residual, self._fused = add_residual, fused
        self._stream = torch.cuda.Stream(device)
        with torch.cuda.stream(self._stream):
            llama_mlp_combined_ops(self.attn_output, self.residual, *args, **kwargs)  # eager: workspace, code objects
            self.residual.zero_()
            torch.cuda.synchronize(device)
            self.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(self.graph, stream=self._stream):
                self.mlp_output, residual_out = llama_mlp_combined_ops(self.attn_output, self.residual, *args, **kwargs)
        assert residual_out.data_ptr() == self.residual.data_ptr()  # updated in place
        # a call allocates nothing and needs no workspace of the stream it is made on, as a replay
        self._memory = _block_memory(rows, hidden, gate_up_weight, down_weight, device) if fused else None
        torch.cuda.synchronize(device)

    def __call__(self, attn_output: Tensor, residual: Tensor) -> Tuple[Tensor, Tensor]:
        """The block on these inputs; returns (mlp_output, residual), this object's buffers, with the inputs' sum and a copy of the first input in
        them as a replay leaves them.

        What the native block does not take (inputs to convert, to broadcast or to copy) is copied in and replayed.  In a loop, us, with two
        copies and a replay / the replay alone / this way: 8 rows of 4096 x 14336 43.0 / 38.9 / 32.2, on six objects in turn, which
        reads every weight from memory, 44.3 / 40.2 / 33.6; one row of 2048 x 6144 34.4 / 22.6 / 15.0 and 34.9 / 23.1 / 16.4.  Starting a graph
        costs the GPU about 6 us more than the launches in it."""
        if self._fused and runs_now(attn_output) and not torch.cuda.is_current_stream_capturing():
            if _native_block(attn_output, residual, self.residual, self.attn_output, self.mlp_output, *self._operands, self._add_residual,
                             self._memory):
                return self.mlp_output, self.residual
        self.attn_output.copy_(attn_output)
        self.residual.copy_(residual)
        self.graph.replay()
        return self.mlp_output, self.residual
