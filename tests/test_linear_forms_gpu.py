"""`apply_fp8_linear` takes the same forms of its arguments, and refuses the same ones, at every row count: one skinny GEMM (5, 40),
two of them or one tiled GEMM (40 with k = 528), one tiled GEMM (65, 130)."""
import pytest
import torch

import hf_rocm_kernels
from hf_rocm_kernels.layers import apply_fp8_linear
from hf_rocm_kernels.utils.fp8 import amax_scale, fp8_quantize

pytestmark = pytest.mark.gpu
N = 264
SIZES = [(5, 512), (40, 512), (40, 528), (65, 512), (130, 528)]


def _operands(m, k):
    torch.manual_seed(m + k)
    w = torch.randn(N, k, device="cuda") * 0.02
    sw = amax_scale(w, dim=1)
    return torch.randn(m, k, device="cuda").to(torch.bfloat16), fp8_quantize(w, sw)[0], sw.reshape(-1).contiguous()


@pytest.mark.parametrize("m,k", SIZES)
@pytest.mark.parametrize("shape", [(N,), (1, N), (1,), (), "rows", "column"])
def test_a_bias_of_any_shape_that_broadcasts(m, k, shape):
    x, w, sw = _operands(m, k)
    shape = {"rows": (m, N), "column": (m, 1)}.get(shape, shape)
    bias = torch.randn(shape, device="cuda").to(torch.bfloat16)
    want = apply_fp8_linear(x, w, sw, residual=bias.expand(m, N).contiguous())  # one addend per value, added and rounded the same way
    assert torch.equal(apply_fp8_linear(x, w, sw, bias=bias), want)
    assert torch.equal(apply_fp8_linear(x, w, sw, bias=bias.float()), want)


@pytest.mark.parametrize("m,k", SIZES)
def test_a_bias_that_does_not_broadcast_is_refused(m, k):
    x, w, sw = _operands(m, k)
    for shape in ((N - 1,), (N, 1), (m + 1, N)):
        with pytest.raises(RuntimeError):
            apply_fp8_linear(x, w, sw, bias=torch.zeros(shape, device="cuda", dtype=torch.bfloat16))


@pytest.mark.parametrize("m,k", SIZES)
def test_scales_of_a_longer_batch(m, k):
    """A buffer of scales for more rows than the call has (a batch that shrank): the first m belong to it."""
    x, w, sw = _operands(m, k)
    q, sx = hf_rocm_kernels.quantize_fp8(x)
    longer = torch.cat([sx, torch.full((3,), float("nan"), device="cuda")])
    assert torch.equal(apply_fp8_linear(q, w, sw, longer), apply_fp8_linear(q, w, sw, sx))


@pytest.mark.parametrize("m,k", SIZES)
def test_operands_that_do_not_fit_are_refused_alike(m, k):
    x, w, sw = _operands(m, k)
    q, sx = hf_rocm_kernels.quantize_fp8(x)
    for bad in (dict(weight_scale=sw[:-1]), dict(weight_scale=sw.double()), dict(input_scale=sx[:3]), dict(input_scale=sx.double()),
                dict(residual=torch.zeros(m, N, device="cuda", dtype=torch.float16)), dict(out_dtype=torch.float32), dict(weight=w[:, :256])):
        with pytest.raises(AssertionError):
            apply_fp8_linear(**{**dict(input=q, weight=w, weight_scale=sw, input_scale=sx), **bad})


@pytest.mark.parametrize("m", [5, 65])
def test_rows_further_apart_than_an_int_counts_are_refused(m):
    k, stride = 512, (1 << 32) + 512  # as an int: 512, the stride of other rows
    x = torch.randn(m, k, device="cuda").to(torch.bfloat16)
    storage = torch.zeros(stride + k, dtype=torch.uint8, device="cuda").view(torch.float8_e4m3fn)
    w, sw = storage.as_strided((2, k), (stride, 1)), torch.ones(2, device="cuda")
    q, sx = hf_rocm_kernels.quantize_fp8(x)
    for call in (lambda: apply_fp8_linear(x, w, sw), lambda: hf_rocm_kernels.skinny_gemm_scaled(q, w.t(), sx, sw),
                 lambda: hf_rocm_kernels.skinny_gemm(q, w.t(), sw[:1])):
        with pytest.raises(RuntimeError):
            call()
