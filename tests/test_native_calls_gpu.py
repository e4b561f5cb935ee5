"""`Fp8Linear` / `apply_fp8_linear` and `skinny_gemm` as one native operator against the operator-by-operator path they replace
(same kernels: same bits), and the calls the operator leaves to that path."""
import itertools

import pytest
import torch

import hf_rocm_kernels
from hf_rocm_kernels.layers import Fp8Linear, apply_fp8_linear, fp8_linear
from hf_rocm_kernels.operators.skinny_gemm import wrapped
from hf_rocm_kernels.utils.fp8 import amax_scale, fp8_quantize
from hf_rocm_kernels.utils.weight_format import pack_weight
from test_gemm_gpu import oracle_checker

pytestmark = pytest.mark.gpu


def _general(monkeypatch):
    monkeypatch.setattr(fp8_linear, "_fp8_linear", lambda *args: None)
    monkeypatch.setattr(wrapped, "_skinny_gemm_new", lambda *args: None)
    monkeypatch.setattr(wrapped, "_skinny_gemm_into", lambda *args: False)


def _bits(t):
    return t.contiguous().view(torch.uint8)


@pytest.mark.parametrize("rows", [1, 5, 17, 64, 65, 130])
@pytest.mark.parametrize("n,k", [(1024, 512), (515, 1024), (2304, 4096)])
def test_linear_same_bits_as_the_general_path(rows, n, k, monkeypatch):
    torch.manual_seed(rows * 1000 + n)
    w = torch.randn(n, k, device="cuda") * 0.02
    sw = amax_scale(w, dim=1)
    q = fp8_quantize(w, sw)[0]
    sw = sw.reshape(-1).contiguous()
    wide = torch.zeros(n, k + 256, device="cuda").to(q.dtype)
    wide[:, :k].copy_(q)  # rows further apart than k
    weights = [(q, sw), (q, sw[:1].clone()), (pack_weight(q), sw), (pack_weight(q, sw), None), (wide[:, :k], sw)]
    for dtype, (weight, scale) in itertools.product((torch.bfloat16, torch.float16), weights):
        x = torch.randn(rows, k, device="cuda").to(dtype)
        x8, sx = hf_rocm_kernels.quantize_fp8(x)
        static = (x.abs().amax().float() / 448).reshape(1)
        bias, residual = torch.randn(n, device="cuda").to(dtype), torch.randn(rows, n, device="cuda").to(dtype)
        calls = [dict(input=x), dict(input=x.view(1, rows, k), input_scale=static), dict(input=x, bias=bias), dict(input=x, residual=residual),
                 dict(input=x8, input_scale=sx, out_dtype=dtype), dict(input=x8, input_scale=static, residual=residual, out_dtype=dtype),
                 dict(input=x, bias=bias, residual=residual), dict(input=x.t().contiguous().t(), bias=bias)]
        got = [apply_fp8_linear(weight=weight, weight_scale=scale, **c) for c in calls]
        with monkeypatch.context() as patch:
            _general(patch)
            want = [apply_fp8_linear(weight=weight, weight_scale=scale, **c) for c in calls]
        for g, w_ in zip(got, want):
            assert g.shape == w_.shape and g.dtype == w_.dtype and torch.equal(_bits(g), _bits(w_))


@pytest.mark.parametrize("m", [32, 33, 48, 64])
@pytest.mark.parametrize("n,k", [(64, 272), (515, 1040), (4104, 1936), (1000, 4112)])
def test_rows_33_to_64_with_a_cut_last_chunk_match_the_oracle(m, n, k, monkeypatch):
    g = torch.Generator().manual_seed(m + n)
    a, w = torch.randn(m, k, generator=g), torch.randn(n, k, generator=g) * 0.02
    sa, sw = amax_scale(a, dim=1), amax_scale(w, dim=1)
    a, w, sa, sw = fp8_quantize(a, sa)[0], fp8_quantize(w, sw)[0], sa.reshape(-1), sw.reshape(-1)
    bias = torch.randn(n, generator=g).to(torch.bfloat16)
    for b in (None, bias):
        check = oracle_checker(a, w.t(), sa, sw, torch.bfloat16, base=None if b is None else b.expand(m, n).contiguous())
        args = a.cuda(), w.cuda(), sw.cuda(), sa.cuda(), None if b is None else b.cuda()
        native = apply_fp8_linear(*args)
        check(native)
        with monkeypatch.context() as patch:
            _general(patch)
            assert torch.equal(native, apply_fp8_linear(*args))


@pytest.mark.parametrize("m,n,k", [(1, 4096, 4096), (7, 514, 512), (33, 1024, 2304), (64, 130, 256), (3, 512, 384)])
def test_skinny_gemm_same_bits_as_the_general_path(m, n, k, monkeypatch):
    torch.manual_seed(m)
    a = torch.randn(m, k, device="cuda").to(torch.float8_e4m3fn)
    b = torch.randn(n, k, device="cuda").to(torch.float8_e4m3fn).t()
    scale = torch.tensor([0.013], device="cuda")
    base = torch.randn(m, n, device="cuda").to(torch.bfloat16)
    got = hf_rocm_kernels.skinny_gemm(a, b, scale), hf_rocm_kernels.skinny_gemm(a, b, scale, base.clone())
    _general(monkeypatch)
    want = hf_rocm_kernels.skinny_gemm(a, b, scale), hf_rocm_kernels.skinny_gemm(a, b, scale, base.clone())
    for g, w in zip(got, want):
        assert g.dtype == w.dtype and torch.equal(g, w)


def test_refused_calls_are_refused_as_before():
    a = torch.zeros(4, 512, device="cuda").to(torch.float8_e4m3fn)
    b = torch.zeros(64, 512, device="cuda").to(torch.float8_e4m3fn)
    one = torch.ones(1, device="cuda")
    for bad in (lambda: hf_rocm_kernels.skinny_gemm(a, b, one), lambda: hf_rocm_kernels.skinny_gemm(a, b.t(), one.double()),
                lambda: hf_rocm_kernels.skinny_gemm(a, b.t(), one, torch.zeros(4, 63, device="cuda", dtype=torch.float16)),
                lambda: hf_rocm_kernels.skinny_gemm(a, b.t(), one.cpu()), lambda: apply_fp8_linear(a, b, one),
                lambda: apply_fp8_linear(torch.zeros(4, 512, device="cuda"), b, one),
                lambda: apply_fp8_linear(torch.zeros(4, 512, device="cuda").half(), b, None)):
        with pytest.raises(AssertionError):
            bad()
    with pytest.raises(RuntimeError):
        hf_rocm_kernels.skinny_gemm(a, b[:63].t(), one)  # an odd number of columns


def test_linear_outputs_carry_no_autograd_history_and_keep_leading_dimensions():
    layer = Fp8Linear.from_float(torch.nn.Linear(512, 256, device="cuda", dtype=torch.float16))
    x = torch.randn(2, 3, 512, device="cuda", dtype=torch.float16, requires_grad=True)
    y = layer(x)
    assert y.shape == (2, 3, 256) and not y.requires_grad
    assert layer(x[:0]).shape == (0, 3, 256)


@pytest.mark.parametrize("rows", [4, 80])
def test_recorded_and_batched_calls_go_the_general_way(rows):
    """A trace that held a whole-call operator would replay it on inputs it does not take, and get nothing back."""
    from torch.fx.experimental.proxy_tensor import make_fx
    layer = Fp8Linear.from_float(torch.nn.Linear(512, 256, device="cuda", dtype=torch.float16))
    x = torch.randn(rows, 512, device="cuda", dtype=torch.float16)
    for pre_dispatch in (False, True):
        graph = make_fx(lambda a: layer(a), pre_dispatch=pre_dispatch)(x)
        names = [str(node.target) for node in graph.graph.nodes]
        assert any("quantize_fp8" in name for name in names) and not any("fp8_linear" in name for name in names)
        assert torch.equal(graph(x), layer(x))
    with pytest.raises(RuntimeError):
        torch.jit.trace(layer, x, check_trace=False)
    with pytest.raises(RuntimeError):
        torch.vmap(layer)(x.view(2, rows // 2, 512))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,cols", [(1, 8), (3, 2050), (5, 14648), (130, 4096), (2, 32768), (2, 40960)])
def test_row_kernels_same_bits_as_the_general_path(rows, cols, dtype, monkeypatch):
    from hf_rocm_kernels.operators.residual_rms import wrapped as rms
    from hf_rocm_kernels.operators.swiglu import wrapped as swi
    gen = torch.Generator(device="cuda").manual_seed(rows + cols)
    x, res = (torch.randn(rows, cols, generator=gen, device="cuda").to(dtype) for _ in range(2))
    w = torch.randn(cols, generator=gen, device="cuda").to(dtype)
    both = torch.randn(rows, 2 * cols, generator=gen, device="cuda").to(dtype)
    scale = torch.tensor([0.02], device="cuda")
    calls = [lambda r: rms.residual_rms(x, r, w, 1e-5, scale), lambda r: rms.residual_rms(x, r, w, 1e-5), lambda r: (swi.swiglu(both, scale),)]
    if cols % 8 == 0 and cols <= 32768:
        calls += [lambda r: rms.residual_rms_dynamic(x, r, w, 1e-5), lambda r: swi.swiglu_dynamic(both)]
    for call in calls:
        native = call(res.clone())
        with monkeypatch.context() as patch:
            patch.setattr(rms, "_residual_rms_new", lambda *args: None)
            patch.setattr(swi, "_swiglu_new", lambda *args: None)
            patch.setattr(rms, "_residual_rms_dynamic_new", lambda *args: (None, None))
            patch.setattr(swi, "_swiglu_dynamic_new", lambda *args: (None, None))
            general = call(res.clone())
        assert len(native) == len(general)
        for got, want in zip(native, general):
            assert got.shape == want.shape and got.dtype == want.dtype and torch.equal(_bits(got), _bits(want))


def test_row_kernels_refuse_what_they_refused():
    from hf_rocm_kernels import residual_rms, residual_rms_dynamic, swiglu, swiglu_dynamic
    x, w, one = torch.zeros(4, 512, device="cuda", dtype=torch.bfloat16), torch.ones(512, device="cuda", dtype=torch.bfloat16), torch.ones(1, device="cuda")
    keep = x.clone()
    for call in (lambda: residual_rms(x, x[:2], w, 1e-5, one), lambda: residual_rms(x, x.clone(), w[:256], 1e-5, one), lambda: residual_rms(x, x.clone().half(), w, 1e-5, one),
                 lambda: residual_rms(x.t(), x.t().clone(), w[:4], 1e-5, one), lambda: residual_rms(x, x.clone(), w, 0.0, one), lambda: residual_rms(x, x.cpu(), w, 1e-5, one),
                 lambda: residual_rms(x, x.clone(), w, 1e-5, one.cpu()), lambda: residual_rms(x.float(), x.float(), w, 1e-5, one),
                 lambda: residual_rms_dynamic(x[:, :508].contiguous(), x[:, :508].contiguous(), w[:508], 1e-5), lambda: swiglu(x[:, :511].contiguous(), one),
                 lambda: swiglu(x.t(), one), lambda: swiglu(x, torch.ones(2, device="cuda")), lambda: swiglu_dynamic(x[:, :24].contiguous())):
        with pytest.raises(AssertionError):
            call()
    with pytest.raises(RuntimeError):
        swiglu(x, one.half())
    assert torch.equal(x, keep)
    # a tensor that autograd follows is taken, as it always was
    weight = w.clone().requires_grad_()
    got, want = residual_rms(x, x.clone(), weight, 1e-5, one), residual_rms(x, x.clone(), w, 1e-5, one)
    assert torch.equal(_bits(got[0]), _bits(want[0]))
    with torch.inference_mode():
        assert torch.equal(_bits(swiglu(x, one)), _bits(swiglu(x.clone(), one)))


@pytest.mark.parametrize("rows", [0, 3])
def test_row_kernels_take_tensors_that_require_a_gradient_and_empty_batches(rows, monkeypatch):
    """Such calls run as the native operator at once; the general way behind a refusal of it took them longer than it alone."""
    from hf_rocm_kernels.operators.residual_rms import wrapped as rms
    from hf_rocm_kernels.operators.swiglu import wrapped as swi
    x, res, w = (torch.randn(*shape, device="cuda", dtype=torch.bfloat16) for shape in ((rows, 512), (rows, 512), (512,)))
    scale = torch.tensor([0.02], device="cuda")
    calls = {"static": lambda x, r, w: rms.residual_rms(x, r, w, 1e-5, scale), "16 bits": lambda x, r, w: rms.residual_rms(x, r, w, 1e-5),
             "dynamic": lambda x, r, w: rms.residual_rms_dynamic(x, r, w, 1e-5), "swiglu": lambda x, r, w: (swi.swiglu(x, scale),),
             "swiglu dynamic": lambda x, r, w: swi.swiglu_dynamic(x)}
    with monkeypatch.context() as patch:  # the general way
        patch.setattr(rms, "runs_now", lambda t: False)
        patch.setattr(swi, "runs_now", lambda t: False)
        want = {name: call(x, res.clone(), w) for name, call in calls.items()}
    monkeypatch.setattr(rms, "residual_rms_checks", None)  # the general way ends here
    monkeypatch.setattr(swi, "swiglu_checks", None)
    for x_, w_ in ((x, w), (x, torch.nn.Parameter(w.clone())), (x.clone().requires_grad_(), w)):
        for name, call in calls.items():
            got = call(x_, res.clone(), w_)
            for g, t in zip(got, want[name]):
                assert g.shape == t.shape and g.dtype == t.dtype and not g.requires_grad and torch.equal(_bits(g), _bits(t)), name
