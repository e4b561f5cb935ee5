"""The fused MLP block as one native operator against the launches of its wrappers (same kernels: same bits), and the calls it leaves
to them."""
import itertools
import sys

import pytest
import torch

from hf_rocm_kernels.combined_ops.llama_mlp import LlamaMlpGraph, llama_mlp_combined_ops
from hf_rocm_kernels.utils.weight_format import pack_weight
from test_gemm_gpu import all_plans

pytestmark = pytest.mark.gpu
MODULE = sys.modules["hf_rocm_kernels.combined_ops.llama_mlp"]


def _block(hidden, inter, dtype, packed=(False, False), wide=0, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    w1 = (torch.randn((2 * inter, hidden + wide), generator=gen, device="cuda") * 4).to(torch.float8_e4m3fn)[:, :hidden]
    w2 = (torch.randn((hidden, inter + wide), generator=gen, device="cuda") * 4).to(torch.float8_e4m3fn)[:, :inter]
    norm = (1 + 0.1 * torch.randn(hidden, generator=gen, device="cuda")).to(dtype)
    s = [torch.tensor([v], device="cuda") for v in (0.013, 0.0005, 0.01, 0.0004)]
    return (norm, 1e-5, pack_weight(w1) if packed[0] else w1.t(), s[0], s[1], pack_weight(w2) if packed[1] else w2.t(), s[2], s[3])


def _rows(m, hidden, dtype, seed=1):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn((m, hidden), generator=gen, device="cuda").to(dtype) for _ in range(2)]


def _same(got, want):
    assert all(g.dtype == w.dtype and torch.equal(g.view(torch.int16), w.view(torch.int16)) for g, w in zip(got, want))


def _counted(monkeypatch):
    taken = []
    native = MODULE._llama_mlp
    monkeypatch.setattr(MODULE, "_llama_mlp", lambda *a: taken.append(native(*a)) or taken[-1])
    return taken


@pytest.mark.parametrize("m", [1, 8, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("hidden,inter", [(256, 512), (1280, 1024), (2048, 2816), (4096, 1536), (8192, 8448)])
def test_same_bits_as_the_wrappers(m, hidden, inter, monkeypatch):
    taken = _counted(monkeypatch)
    for dtype, packed, wide in ((torch.bfloat16, (False, False), 0), (torch.float16, (True, True), 0), (torch.bfloat16, (True, False), 0),
                                (torch.float16, (False, False), 64)):
        args = _block(hidden, inter, dtype, packed, wide)
        x, res = _rows(m, hidden, dtype)
        for add in (True, False):
            r1, r2 = res.clone(), res.clone()
            got = llama_mlp_combined_ops(x, r1, *args, add_residual=add, fused=True)
            with monkeypatch.context() as patch:
                patch.setattr(MODULE, "_llama_mlp", lambda *a: False)
                want = llama_mlp_combined_ops(x, r2, *args, add_residual=add, fused=True)
            assert got[1] is r1
            _same(got, want)
    assert taken == [True] * 8


@pytest.mark.parametrize("m,hidden,inter", [(1, 2048, 2816), (8, 4096, 1536), (40, 1280, 1024), (3, 16640, 512), (2, 32768, 512)])
def test_graph_call_leaves_what_copies_and_a_replay_leave(m, hidden, inter, monkeypatch):
    taken = _counted(monkeypatch)
    args = _block(hidden, inter, torch.bfloat16)
    block, plain = LlamaMlpGraph(m, hidden, *args), LlamaMlpGraph(m, hidden, *args)
    del taken[:]
    other = torch.cuda.Stream()

    def both(make):
        got = block(*make(block))
        a, r = make(plain)
        plain.attn_output.copy_(a)
        plain.residual.copy_(r)
        plain.graph.replay()
        torch.cuda.synchronize()
        _same((*got, block.attn_output), (plain.mlp_output, plain.residual, plain.attn_output))
        assert got[0] is block.mlp_output and got[1] is block.residual

    x, res = _rows(m, hidden, torch.bfloat16)
    before = x.clone(), res.clone()
    both(lambda b: (x, res))
    assert torch.equal(x, before[0]) and torch.equal(res, before[1])
    both(lambda b: (b.mlp_output, b.residual))     # a chain of blocks
    both(lambda b: (x, b.mlp_output))
    both(lambda b: (b.residual, res))
    both(lambda b: (b.attn_output, b.residual))
    torch.cuda.synchronize()
    with torch.cuda.stream(other):
        both(lambda b: (res, x))
    assert taken == [True] * 6
    both(lambda b: (x, b.attn_output))             # the copy of the input would come first
    both(lambda b: (x.float(), res))               # converted by copy_
    both(lambda b: (x.t().contiguous().t(), res))
    both(lambda b: (x[:1], res))                   # broadcast
    assert taken[6:] == [False, False, m == 1, m == 1]  # (one row is contiguous either way)
    block.graph.replay()                           # the graph itself still runs on its buffers
    plain.graph.replay()
    _same((block.mlp_output, block.residual), (plain.mlp_output, plain.residual))


def test_calls_that_are_left_to_the_wrappers(monkeypatch):
    """Nothing may have been written by then: the wrappers add the residual themselves, or refuse."""
    taken = _counted(monkeypatch)
    hidden, inter = 512, 1024
    args = _block(hidden, inter, torch.bfloat16)
    x, res = _rows(4, hidden, torch.bfloat16)
    storage = torch.zeros(4 * hidden + 4, dtype=torch.bfloat16, device="cuda")
    odd = storage[4:].view(4, hidden)  # 8-byte, not 16-byte aligned: the RMSNorm takes its element-wise way
    odd.copy_(res)
    got = llama_mlp_combined_ops(x, odd, *args, add_residual=True, fused=True)
    want = llama_mlp_combined_ops(x, res.clone(), *args, add_residual=True, fused=True)
    assert taken == [False, True] and torch.equal(odd, want[1]) and torch.allclose(got[0].float(), want[0].float(), rtol=0.05, atol=0.5)
    for change, error in itertools.chain([({1: 0.0}, AssertionError), ({3: args[3].cpu()}, (AssertionError, RuntimeError)), ({4: args[4].double()}, AssertionError),
                                          ({6: args[6].repeat(2)}, AssertionError), ({0: args[0][:-8]}, AssertionError), ({5: args[5][:-256]}, AssertionError)]):
        bad = tuple(change.get(i, a) for i, a in enumerate(args))
        with pytest.raises(error):
            llama_mlp_combined_ops(x, res.clone(), *bad, add_residual=True, fused=True)
    assert not any(taken[2:])


def test_results_that_overlap_are_not_written():
    hidden = 512
    norm, eps, w1, s1, s2, w2, s3, s4 = _block(hidden, 1024, torch.bfloat16)
    x, res = _rows(4, hidden, torch.bfloat16)
    out, before = torch.zeros_like(x), (x.clone(), res.clone())
    half = torch.zeros(6 * hidden, dtype=torch.bfloat16, device="cuda")
    for residual_out, copy, output in ((res, None, res), (res, res, out), (out, None, out), (half[:4 * hidden].view(4, hidden), half[2 * hidden:].view(4, hidden), out)):
        assert not MODULE._llama_mlp(x, res, residual_out, copy, norm, eps, w1, -1, s1, s2, w2, -1, s3, s4, True, output)
        torch.cuda.synchronize()
        assert torch.equal(x, before[0]) and torch.equal(res, before[1]) and not out.any() and not half.any()


@pytest.mark.parametrize("m,packed", [(8, False), (16, True), (64, False), (64, True)])
def test_graph_call_takes_no_memory_and_no_workspace(m, packed, monkeypatch):
    """As a replay: the object holds what its calls need, also on a stream that has launched nothing before."""
    from hf_rocm_kernels import _capi
    lib, taken = _capi.load(), _counted(monkeypatch)
    hidden, inter = 1024, 5120
    args = _block(hidden, inter, torch.bfloat16, (packed, packed))
    block = LlamaMlpGraph(m, hidden, *args)
    rows = [_rows(m, hidden, torch.bfloat16, seed) for seed in range(4)]
    want = [[t.clone() for t in llama_mlp_combined_ops(x, res.clone(), *args, add_residual=True, fused=True)] for x, res in rows]
    assert lib.hfrk_llama_mlp_workspace_bytes(64, hidden, inter, 0, 0) > 0  # k is split between workgroups in one of the two
    torch.cuda.synchronize()
    del taken[:]
    for stream in [torch.cuda.Stream() for _ in range(3)]:
        if lib.hfrk_workspace_id(stream.cuda_stream) >= 0:
            continue  # a handle that an earlier test's stream had
        for (x, res), expected in zip(rows, want):
            before = torch.cuda.memory_stats()["allocation.all.allocated"]
            with torch.cuda.stream(stream):
                got = block(x, res)
            assert torch.cuda.memory_stats()["allocation.all.allocated"] == before
            torch.cuda.synchronize()
            _same(got, expected)
        assert lib.hfrk_workspace_id(stream.cuda_stream) == -1
    assert taken and all(taken)


def test_graph_call_whose_plan_has_grown_replays(monkeypatch):
    import ctypes
    from hf_rocm_kernels import _capi
    lib, taken = _capi.load(), _counted(monkeypatch)
    m, hidden, inter = 8, 1024, 5120
    args = _block(hidden, inter, torch.bfloat16)
    block = LlamaMlpGraph(m, hidden, *args)
    x, res = _rows(m, hidden, torch.bfloat16)
    want = [t.clone() for t in block(x, res)]
    assert lib.hfrk_llama_mlp_workspace_bytes(m, hidden, inter, 0, 0) == 0
    plan = next(p for p in all_plans(m, hidden, inter) if p.wn > 0)  # partial sums between workgroups
    try:
        assert lib.hfrk_plan_table_set(m, hidden, inter, 0, ctypes.byref(plan)) == 0
        assert lib.hfrk_llama_mlp_workspace_bytes(m, hidden, inter, 0, 0) > 0
        got = block(x, res)
        torch.cuda.synchronize()
        assert taken[-1] is False
        _same(got, want)
    finally:
        lib.hfrk_plan_table_set(m, hidden, inter, 0, None)
    block(x, res)
    assert taken[-1] is True


def test_graph_call_is_refused_while_a_caller_captures():
    """A graph is not replayed into another; what can be captured is llama_mlp_combined_ops."""
    args = _block(512, 1024, torch.bfloat16)
    block = LlamaMlpGraph(4, 512, *args)
    x, res = _rows(4, 512, torch.bfloat16)
    want = [t.clone() for t in block(x, res)]
    with pytest.raises(RuntimeError):
        with torch.cuda.graph(torch.cuda.CUDAGraph(), stream=torch.cuda.Stream()):
            block(x, res)
    torch.cuda.synchronize()
    _same(block(x, res), want)


def test_a_meta_tensor_is_refused():
    hidden = 512
    args = _block(hidden, 1024, torch.bfloat16)
    block = LlamaMlpGraph(4, hidden, *args)
    x, res = _rows(4, hidden, torch.bfloat16)
    with pytest.raises(AssertionError):
        llama_mlp_combined_ops(x, res.to("meta"), *args, add_residual=True, fused=True)
    with pytest.raises(AssertionError):
        llama_mlp_combined_ops(x, res, args[0], 1e-5, args[2].to("meta"), *args[3:], add_residual=True, fused=True)
    with pytest.raises((RuntimeError, NotImplementedError)):
        block(x, res.to("meta"))
