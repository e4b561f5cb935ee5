"""Whether a call may go to an operator that answers "not one of mine" at run time."""
import torch
from torch import Tensor

from hf_rocm_kernels._HFRK_C import nothing_intercepts

_is_compiling = torch.compiler.is_compiling


def runs_now(t: Tensor) -> bool:
    """True for a GPU tensor in a call that runs here and now.  Under a compiler, a tracer (torch.jit.trace and pre-dispatch tracing
    among them), a functorch transform, a fake-tensor or another dispatch mode, or with a tensor subclass, such an operator's answer is
    not known or would be recorded for calls it does not take: those go the general way, whose operators check their arguments."""
    return t.is_cuda and type(t) is Tensor and not _is_compiling() and nothing_intercepts()
