"""The operators trace with fake tensors: every wrapper runs under FakeTensorMode without a GPU and returns outputs of
the right shape and dtype (no kernel runs, no device is touched)."""
import pytest
import torch
from torch._subclasses import FakeTensorMode

import hf_rocm_kernels
from hf_rocm_kernels.combined_ops.llama_mlp import llama_mlp_combined_ops
from hf_rocm_kernels.layers import apply_fp8_linear

FP8 = torch.float8_e4m3fn


def _fp8(*shape):
    return torch.empty(*shape, device="cuda", dtype=FP8)


def test_every_operator_has_a_fake_implementation():
    from hf_rocm_kernels import _fake_kernels
    names = set(_fake_kernels._RETURNS_NOTHING) | set(_fake_kernels._RETURNS_STATUS)
    defined = {n.split("::")[1].split(".")[0] for n in torch._C._dispatch_get_all_op_names() if n.startswith("_HFRK_C::")}
    assert defined == names


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_wrappers_under_fake_tensors(dtype):
    with FakeTensorMode():
        m, hidden, inter = 8, 4096, 14336
        one = torch.empty(1, device="cuda")
        x = torch.empty(m, hidden, device="cuda", dtype=dtype)
        res = torch.empty_like(x)
        w = torch.empty(hidden, device="cuda", dtype=dtype)

        q, res2 = hf_rocm_kernels.residual_rms(input=x, residual=res, weight=w, epsilon=1e-5, scale_tensor=one)
        assert q.shape == (m, hidden) and q.dtype == FP8 and res2.shape == res.shape
        q, _, scales = hf_rocm_kernels.residual_rms_dynamic(input=x, residual=res, weight=w, epsilon=1e-5)
        assert q.dtype == FP8 and scales.shape == (m,)

        gate_up_w = _fp8(2 * inter, hidden)
        proj = hf_rocm_kernels.skinny_gemm(q, gate_up_w.t(), one, output=torch.empty(m, 2 * inter, device="cuda", dtype=dtype))
        assert proj.shape == (m, 2 * inter) and proj.dtype == dtype
        act = hf_rocm_kernels.swiglu(gate_up_proj=proj, scale_tensor=one)
        assert act.shape == (m, inter) and act.dtype == FP8
        act, act_scales = hf_rocm_kernels.swiglu_dynamic(proj)[:2]
        assert act.shape == (m, inter) and act_scales.shape == (m,)

        down_w = _fp8(hidden, inter)
        out = hf_rocm_kernels.skinny_gemm_scaled(act, down_w.t(), act_scales, torch.empty(hidden, device="cuda"))
        assert out.shape == (m, hidden) and out.dtype == torch.bfloat16
        out = hf_rocm_kernels.skinny_gemm_add(act, down_w.t(), one, None, base=res)
        assert out.shape == (m, hidden)
        fused = hf_rocm_kernels.skinny_gemm_swiglu(q, gate_up_w.t(), one, None, one, intermediate_dtype=dtype)
        assert fused.shape == (m, inter) and fused.dtype == FP8

        q, s = hf_rocm_kernels.quantize_fp8(x)
        assert q.shape == x.shape and q.dtype == FP8 and s.shape == (m,)
        y = apply_fp8_linear(x, down_w[:, :hidden].contiguous(), torch.empty(hidden, device="cuda"))
        assert y.shape == (m, hidden) and y.dtype == dtype


@pytest.mark.parametrize("fused", [False, True])
def test_mlp_chain_under_fake_tensors(fused):
    with FakeTensorMode():
        m, hidden, inter = 4, 4096, 14336
        one = torch.empty(1, device="cuda")
        x = torch.empty(m, hidden, device="cuda", dtype=torch.bfloat16)
        out, res = llama_mlp_combined_ops(x, torch.empty_like(x), torch.empty(hidden, device="cuda", dtype=torch.bfloat16), 1e-5,
                                          _fp8(2 * inter, hidden).t(), one, one, _fp8(hidden, inter).t(), one, one,
                                          add_residual=True, fused=fused)
        assert out.shape == (m, hidden) and out.dtype == torch.bfloat16 and res.shape == (m, hidden)


class _Block(torch.nn.Module):
    def __init__(self):
        super().__init__()
        self.gate_up = torch.nn.Linear(512, 1024, bias=False)
        self.down = torch.nn.Linear(512, 512, bias=True)
        self.odd = torch.nn.Linear(100, 8)        # in_features not a multiple of 256: stays
        self.lm_head = torch.nn.Linear(512, 64)   # skipped by name
        self.inner = torch.nn.Sequential(torch.nn.Linear(256, 256), torch.nn.ReLU())


def test_convert_linear_layers_and_state_dict_round_trip_on_the_cpu():
    """Conversion and (de)serialisation are host work: which layers are replaced, what the state dict holds, and that
    a freshly converted model takes another one's state."""
    from hf_rocm_kernels.layers import Fp8Linear, convert_linear_layers
    from oracle import fp8 as ofp8
    torch.manual_seed(0)
    model = _Block().to(torch.bfloat16)
    float_weight = model.down.weight.detach().clone()
    assert convert_linear_layers(model, skip=("lm_head",)) == 3
    assert isinstance(model.gate_up, Fp8Linear) and isinstance(model.down, Fp8Linear) and isinstance(model.inner[0], Fp8Linear)
    assert type(model.odd) is torch.nn.Linear and type(model.lm_head) is torch.nn.Linear
    assert convert_linear_layers(model) == 1          # a second pass finds only lm_head left
    # the quantised weight is the oracle's quantisation with per-channel amax/448 scales
    scale = ofp8.amax_scale(float_weight, dim=1)
    want, _ = ofp8.fp8_quantize(float_weight, scale)
    assert torch.equal(model.down.weight_data.view(torch.uint8), want.view(torch.uint8))
    assert torch.equal(model.down.weight_scale, scale.reshape(-1))
    state = model.state_dict()
    assert state["down.weight_data"].dtype == FP8 and state["down.weight_scale"].shape == (512,) and "gate_up.bias" not in state
    other = _Block().to(torch.bfloat16)
    convert_linear_layers(other)
    result = other.load_state_dict(state)
    assert not result.missing_keys and not result.unexpected_keys
    for name in ("gate_up", "down", "lm_head"):
        a, b = getattr(model, name), getattr(other, name)
        assert torch.equal(a.weight_data.view(torch.uint8), b.weight_data.view(torch.uint8)) and torch.equal(a.weight_scale, b.weight_scale)
        assert b.weight is b.weight_data and not b.packed
    assert "weight=row-major" in repr(other.down)


def test_a_traced_call_records_operators_that_check_their_arguments():
    """The whole-call operators return nothing for a call they do not take, so a trace must not hold one, and a call that is
    refused on tensors is refused on fake ones."""
    from torch.fx.experimental.proxy_tensor import make_fx
    with FakeTensorMode():
        x, w, sw = torch.empty(8, 512, device="cuda", dtype=torch.bfloat16), _fp8(256, 512), torch.empty(256, device="cuda")
        graph = make_fx(lambda a: apply_fp8_linear(a, w, sw))(x)
        assert not any("fp8_linear" in str(node.target) for node in graph.graph.nodes)
        with pytest.raises(AssertionError):
            apply_fp8_linear(x, _fp8(256, 768), sw)
        with pytest.raises(AssertionError):
            hf_rocm_kernels.skinny_gemm(_fp8(8, 512), _fp8(256, 768).t(), torch.empty(1, device="cuda"))


def test_whole_call_operators_take_no_meta_tensor_among_others():
    """One meta tensor among tensors with data sends a call to the shape-only implementations; a result of theirs would be one that nobody
    computed.  A call on meta tensors alone asks for shapes."""
    def tensors(device, *others):
        make = lambda i, *shape, dtype=FP8: torch.empty(*shape, device=others[0] if others and i == others[1] else device, dtype=dtype)
        return [make(0, 4, 512, dtype=torch.bfloat16), make(1, 256, 512), make(2, 1, dtype=torch.float32), make(3, 4, 512), make(4, 4, 256, dtype=torch.float16),
                make(5, 512, dtype=torch.bfloat16), make(6, 1024, 512), make(7, 512, 512)]

    ops = torch.ops._HFRK_C
    linear = lambda x, w, one, q, d, norm, gate_up, down: ops.fp8_linear(x, w, -1, one, None, None, None, None)
    new = lambda x, w, one, q, d, norm, gate_up, down: ops.skinny_gemm_new(q, w.t(), one)
    into = lambda x, w, one, q, d, norm, gate_up, down: ops.skinny_gemm_into(q, w.t(), one, d)
    mlp = lambda x, w, one, q, d, norm, gate_up, down: ops.llama_mlp(x, x, x, None, norm, 1e-5, gate_up.t(), -1, one, one, down.t(), -1, one, one, True, x)
    alone = tensors("meta")
    assert linear(*alone).shape == (4, 256) and new(*alone).shape == (4, 256) and into(*alone) is True and mlp(*alone) is True
    for at in (1, 2):
        assert linear(*tensors("cpu", "meta", at)) is None and linear(*tensors("meta", "cpu", at)) is None
        assert new(*tensors("cpu", "meta", at)) is None and into(*tensors("cpu", "meta", at)) is False
    for at in (0, 2, 5, 6, 7):
        assert mlp(*tensors("cpu", "meta", at)) is False


def _interceptors():
    """Ways a call is recorded, batched or replaced: each runs its argument with a tensor."""
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.utils._python_dispatch import TorchDispatchMode

    class Passing(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    def inside(mode, f):
        with mode:
            return f(torch.ones(2, 2))

    ones = torch.ones(2, 2)
    return {
        "jit.trace": lambda f: torch.jit.trace(f, ones, check_trace=False),
        "make_fx": lambda f: make_fx(f)(ones),
        "make_fx before dispatch": lambda f: make_fx(f, pre_dispatch=True)(ones),
        "vmap": lambda f: torch.vmap(f)(ones),
        "jvp": lambda f: torch.func.jvp(f, (ones,), (ones,)),
        "grad": lambda f: torch.func.grad(lambda x: f(x).sum())(ones),
        "functionalize": lambda f: torch.func.functionalize(f)(ones),
        "fake": lambda f: inside(FakeTensorMode(), f),
        "dispatch mode": lambda f: inside(Passing(), f),
    }


@pytest.mark.parametrize("way", sorted(_interceptors()))
def test_whole_call_operators_stay_out_of_calls_that_something_intercepts(way):
    from hf_rocm_kernels._HFRK_C import nothing_intercepts
    seen = []

    def call(x):
        seen.append(nothing_intercepts())
        return x * 2

    assert nothing_intercepts()
    _interceptors()[way](call)
    assert seen and not any(seen)
    assert nothing_intercepts()


def test_settings_that_change_no_call_are_no_interception():
    from hf_rocm_kernels._HFRK_C import nothing_intercepts
    for setting in (torch.no_grad(), torch.inference_mode(), torch.autocast("cpu", dtype=torch.bfloat16), torch.device("cpu"),
                    torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t)):
        with setting:
            assert nothing_intercepts()
