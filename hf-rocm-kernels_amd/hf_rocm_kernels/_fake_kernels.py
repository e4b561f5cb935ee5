"""Shape-only ("fake") implementations of the `_HFRK_C` operators, for tracing.

The reference registers its operators on the CUDA dispatch key only (csrc/torch_bindings.cpp:20-41), so they cannot
be traced with fake tensors.  Every operator here writes into tensors the caller passes (`Tensor!` in the schema)
and returns nothing or a status integer, so the fake implementation has nothing to compute: it returns None, or 0
for the GEMM entry points (the status of a call whose arguments the real implementation accepts).  With these
registered torch can trace through the operators; the mutations are functionalised by torch from the schema.
A tracer cannot keep an operator that returns an integer inside a graph, so while torch is compiling the GEMM
wrappers call `skinny_gemm_checked`, which raises on a non-zero status instead of returning it; with that,
`torch.compile(..., fullgraph=True)` takes the whole MLP block as one graph.  Nothing here runs when an operator
is called on real tensors.
"""
import torch

import hf_rocm_kernels._HFRK_C  # noqa: F401  (registers torch.ops._HFRK_C)

_RETURNS_NOTHING = ("increment", "residual_rms", "swiglu", "pack_weight", "pack_weight_scaled", "unpack_weight", "reencode_fnuz",
                    "residual_rms_dynamic", "swiglu_dynamic", "quantize_fp8", "skinny_gemm_checked", "tiled_gemm")
_RETURNS_STATUS = ("skinny_gemm_tb", "skinny_gemm_scaled", "skinny_gemm_fused", "skinny_gemm_packed", "skinny_gemm_rms_fused",
                   # a result of their own, _OTHER_RESULT; the wrappers keep fake calls away from these (utils/dispatch.py), a caller of
                   # torch.ops need not
                   "fp8_linear", "skinny_gemm_new", "skinny_gemm_into", "llama_mlp", "residual_rms_new", "residual_rms_dynamic_new", "swiglu_new",
                   "swiglu_dynamic_new")


def _nothing(*args, **kwargs) -> None:
    return None


def _success(*args, **kwargs) -> int:
    return 0


def _fp8_linear(input, weight, n, weight_scale, input_scale, bias, residual, out_dtype):
    dtype = out_dtype or (torch.bfloat16 if input.dtype == torch.float8_e4m3fn else input.dtype)
    return input.new_empty((*input.shape[:-1], n if n >= 0 else weight.shape[0]), dtype=dtype)


def _skinny_gemm_new(A, B, scale):
    return A.new_empty((A.shape[0], B.shape[1]), dtype=torch.float16)


def _residual_rms_new(input, residual, weight, epsilon, scale):
    return input.new_empty(input.shape, dtype=input.dtype if scale is None else torch.float8_e4m3fn)


def _residual_rms_dynamic_new(input, residual, weight, epsilon):
    return input.new_empty(input.shape, dtype=torch.float8_e4m3fn), input.new_empty((input.shape[0],), dtype=torch.float32)


def _swiglu_new(gate_up, scale=None):
    return gate_up.new_empty((gate_up.shape[0], gate_up.shape[1] // 2), dtype=torch.float8_e4m3fn)


def _swiglu_dynamic_new(gate_up):
    return _swiglu_new(gate_up), gate_up.new_empty((gate_up.shape[0],), dtype=torch.float32)


def _unless_mixed(answer, refusal):
    """A whole-call operator also lands here when one tensor among device tensors is a meta tensor, which the wrapper's look at its first
    argument does not show: that is no call of the operator's, and the general way refuses it."""
    def fake(*args, **kwargs):
        devices = {a.device.type for a in (*args, *kwargs.values()) if isinstance(a, torch.Tensor)}
        if "meta" in devices and len(devices) > 1:
            return refusal
        return answer(*args, **kwargs)
    return fake


_OTHER_RESULT = {"fp8_linear": _unless_mixed(_fp8_linear, None), "skinny_gemm_new": _unless_mixed(_skinny_gemm_new, None),
                 "skinny_gemm_into": _unless_mixed(lambda A, B, scale, D: True, False), "llama_mlp": _unless_mixed(lambda *args, **kwargs: True, False),
                 "residual_rms_new": _unless_mixed(_residual_rms_new, None), "residual_rms_dynamic_new": _unless_mixed(_residual_rms_dynamic_new, (None, None)),
                 "swiglu_new": _unless_mixed(_swiglu_new, None), "swiglu_dynamic_new": _unless_mixed(_swiglu_dynamic_new, (None, None))}


def register() -> None:
    for name in _RETURNS_NOTHING:
        torch.library.register_fake(f"_HFRK_C::{name}", _nothing)
    for name in _RETURNS_STATUS:
        torch.library.register_fake(f"_HFRK_C::{name}", _OTHER_RESULT.get(name, _success))


register()
