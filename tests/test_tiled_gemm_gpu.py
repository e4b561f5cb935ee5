"""GPU parity of the tiled GEMM (more rows than the skinny kernels take) against the CPU oracle, to the same bar as the skinny
kernels: one output ulp plus 2^-16 of the sum of absolute products.  Every tile shape in both weight layouts, at sizes around
the edges of tiles, stages and splits."""
import ctypes
import os
import subprocess
import sys

import pytest
import torch

from test_gemm_gpu import oracle_checker

pytestmark = pytest.mark.gpu


def _operands(m, n, k, seed):
    from hf_rocm_kernels.utils.fp8 import amax_scale, fp8_quantize
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(m, k, generator=g)
    a[m - 1] *= 20.0
    w = torch.randn(n, k, generator=g) * 0.02
    sa, sw = amax_scale(a, dim=1), amax_scale(w, dim=1)
    return fp8_quantize(a, sa)[0], fp8_quantize(w, sw)[0], sa.reshape(-1), sw.reshape(-1)


# (m, n, k, splits): one row; one tile and one stage; one row and eight columns past a tile, k past a stage and cut unevenly;
# rows of D that are not 16-byte aligned; a last stage cut short; several groups of tiles; fewer stages than the pipeline is deep
SIZES = [(1, 64, 256, 1), (64, 256, 128, 1), (257, 264, 1280, 3), (130, 203, 512, 2), (65, 136, 1008, 1), (600, 520, 768, 1), (200, 72, 16, 1),
         # the 256 x 128 tile on four waves (k no multiple of 128 and 44 stages or more, the last row of tiles more than half full, or many
         # workgroups), and next to it
         (144, 136, 5520, 1), (143, 136, 5520, 1), (144, 136, 5488, 1), (400, 200, 11280, 2), (512, 264, 5520, 1), (512, 264, 2064, 4),
         # several rows and columns of tiles, each with a start in k of its own, over several windows, the last of them shorter
         (600, 520, 5008, 2),
         # two stages a workgroup, the last one cut short
         (600, 520, 400, 2)]


@pytest.mark.parametrize("add", ["none", "bias", "residual"])
@pytest.mark.parametrize("m,n,k,splits", SIZES)
def test_every_tile_shape_matches_the_oracle(m, n, k, splits, add):
    from hf_rocm_kernels import _capi
    from hf_rocm_kernels.utils.weight_format import pack_weight
    lib = _capi.load()
    dtype = torch.float16 if add == "bias" else torch.bfloat16
    a, w, sa, sw = _operands(m, n, k, seed=m + n + k)
    g = torch.Generator().manual_seed(7)
    base = {"none": None, "bias": torch.randn(n, generator=g).to(dtype), "residual": torch.randn(m, n, generator=g).to(dtype)}[add]
    check = oracle_checker(a, w.t(), sa, sw, dtype, base=None if base is None else base.expand(m, n).contiguous())
    dev = [t.cuda() for t in (a, w, sa, sw)]
    dev_base = None if base is None else base.cuda()
    layouts = [(0, dev[1])] + ([(1, pack_weight(dev[1]).data)] if k % 256 == 0 else [])
    for shape in range(5):
        first = None
        for packed, weight in layouts:
            for _ in range(2):
                out = torch.full((m, n), float("nan"), dtype=dtype, device="cuda")
                plan = _capi.TiledPlan(shape, splits, 2 if m > 256 else 1)
                status = lib.hfrk_tiled_gemm(dev[0].data_ptr(), weight.data_ptr(), packed, out.data_ptr(), None if base is None else dev_base.data_ptr(),
                                             n if add == "residual" else 0, dev[2].data_ptr(), 1, dev[3].data_ptr(), 1, m, n, k, k,
                                             _capi.F16 if dtype == torch.float16 else _capi.BF16, ctypes.byref(plan),
                                             torch.cuda.current_stream().cuda_stream)
                _capi.check(status, "hfrk_tiled_gemm")
                torch.cuda.synchronize()
                if first is None:
                    check(out)
                    first = out
                assert torch.equal(out, first), (shape, packed)  # the layouts and repeated launches give the same bits


@pytest.mark.parametrize("m,n,k", [(65, 1000, 2048), (201, 1032, 1040), (300, 4096, 512)])
def test_strided_weights_and_scalar_scales(m, n, k):
    a, w, sa, sw = _operands(m, n, k, seed=3)
    wide = torch.zeros(n, k + 48, dtype=torch.uint8)
    wide[:, :k] = w.view(torch.uint8)
    wide[:, k:] = 0x7F  # NaN beyond the row's end: never read into a sum
    view = wide.cuda().view(torch.float8_e4m3fn)[:, :k]
    out = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
    # Codes reach 448, so sum |a b| over k = 2048 is of the order of 3e6 and its fp32 error bound, 2^-16 of that, of the order of 50:
    # a scale of 0.013 would make that 0.6, beyond the absolute 1e-2 of the check.  2e-6 brings results to order 1.
    one = torch.tensor([2e-6])
    torch.ops._HFRK_C.tiled_gemm(a.cuda(), view.t(), False, n, out, None, one.cuda(), None)
    oracle_checker(a, w.t(), one, torch.ones(1), torch.bfloat16)(out)


def test_argument_errors_and_plans():
    from hf_rocm_kernels import _capi
    lib = _capi.load()
    buf = torch.zeros(1 << 16, dtype=torch.uint8, device="cuda")
    p = buf.data_ptr()

    def call(m=80, n=64, k=128, packed=0, stride=128, dtype=_capi.BF16, plan=None, a=p):
        return lib.hfrk_tiled_gemm(a, p, packed, p + 32768, None, 0, p, 0, None, 0, m, n, k, stride, dtype, plan, None)

    assert call(m=0) == _capi.BAD_SHAPE and call(stride=112) == _capi.BAD_SHAPE
    assert call(k=120, stride=128) == _capi.K_NOT_DIVISIBLE_BY_WARPTILE_K and call(packed=1) == _capi.K_NOT_DIVISIBLE_BY_WARPTILE_K
    assert call(dtype=_capi.FP8_E4M3FN) == _capi.BAD_DTYPE
    assert call(a=p + 8) == _capi.BAD_ALIGNMENT
    for bad in ((5, 1, 1), (-1, 1, 1), (0, 2, 1), (0, 1, 2), (4, 0, 1)):
        assert call(plan=ctypes.byref(_capi.TiledPlan(*bad))) == _capi.INVALID_CONFIG, bad


def test_weights_beyond_the_tiled_kernels_sizes_run_in_pieces():
    from hf_rocm_kernels.layers import apply_fp8_linear
    m, n, k = 66, (1 << 21) + 16, 256
    g = torch.Generator(device="cuda").manual_seed(1)
    a = torch.randint(0, 0x70, (m, k), dtype=torch.uint8, device="cuda", generator=g).view(torch.float8_e4m3fn)
    w = torch.randint(0, 0x70, (n, k), dtype=torch.uint8, device="cuda", generator=g).view(torch.float8_e4m3fn)
    sa, sw = torch.rand(m, device="cuda", generator=g) * 1e-4, torch.full((1,), 1e-2, device="cuda")
    bias = torch.randn(n, device="cuda", generator=g).to(torch.bfloat16)
    whole = apply_fp8_linear(a, w, sw, sa, bias=bias)
    for r0, r1 in ((0, 64), (64, m)):
        assert torch.equal(whole[r0:r1], apply_fp8_linear(a[r0:r1], w, sw, sa[r0:r1], bias=bias))


# (m, n, k) that the skinny entry points hand to the tiled kernel: one tile's height and the smallest row count, ragged columns, k in one and in
# several parts, tiles in pairs on a compute unit
@pytest.mark.parametrize("m,n,k", [(17, 1112, 6912), (64, 3800, 1792), (33, 2136, 15104), (44, 17152, 1792), (64, 1040, 2560)])
def test_skinny_calls_that_run_on_tiles(m, n, k):
    import hf_rocm_kernels as h
    from hf_rocm_kernels import _capi
    from hf_rocm_kernels.utils.weight_format import pack_weight
    lib = _capi.load()
    a, w, sa, sw = _operands(m, n, k, seed=m + n)
    da, dw, dsa, dsw = (t.cuda() for t in (a, w, sa, sw))
    g = torch.Generator().manual_seed(5)
    base = torch.randn(m, n, generator=g).to(torch.bfloat16)
    check = oracle_checker(a, w.t(), sa, sw, torch.bfloat16, base=base)
    outs = []
    for weight in (dw.t(), pack_weight(dw)):
        out = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
        outs.append(h.skinny_gemm_add(da, weight, dsa, dsw, base.cuda(), output=out))
        check(outs[-1])
    for entry in (lib.hfrk_skinny_gemm_ex, lib.hfrk_skinny_gemm_noalloc):  # added to what is there, in place
        out = base.cuda()
        _capi.check(entry(da.data_ptr(), dw.data_ptr(), out.data_ptr(), dsa.data_ptr(), 1, dsw.data_ptr(), 1, m, n, k, k, _capi.BF16, 1, None,
                          torch.cuda.current_stream().cuda_stream), "accumulate")
        torch.cuda.synchronize()
        assert torch.equal(out, outs[0])
    # captured and replayed between other work; the workspace is the capture stream's
    stream, out = torch.cuda.Stream(), torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        h.skinny_gemm_add(da, dw.t(), dsa, dsw, base.cuda(), output=out)
        torch.cuda.synchronize()
        addend, graph = base.cuda(), torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            h.skinny_gemm_add(da, dw.t(), dsa, dsw, addend, output=out)
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, outs[0])
    del graph
    lib.hfrk_release_stream(stream.cuda_stream)
    # rows that are not 16-byte aligned stay where they were
    off = torch.empty(m * n + 4, dtype=torch.bfloat16, device="cuda")[4:].view(m, n)
    off.copy_(base)
    _capi.check(lib.hfrk_skinny_gemm_ex(da.data_ptr(), dw.data_ptr(), off.data_ptr(), dsa.data_ptr(), 1, dsw.data_ptr(), 1, m, n, k, k, _capi.BF16, 1, None,
                                        torch.cuda.current_stream().cuda_stream), "8-byte rows")
    check(off)


# A process of its own: it takes every workspace there is.
_NO_WORKSPACE = """
import ctypes, torch
from hf_rocm_kernels import _capi
lib = _capi.load()
torch.zeros(1, device="cuda")
hip = ctypes.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line))
m, n, k = 65, 64, 4096
a, w = (torch.randn(r, k, device="cuda").to(torch.float8_e4m3fn) for r in (m, n))
one = torch.ones(1, device="cuda")

def call(stream, splits):
    out = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
    plan = ctypes.byref(_capi.TiledPlan(4, splits, 1)) if splits else None
    status = lib.hfrk_tiled_gemm(a.data_ptr(), w.data_ptr(), 0, out.data_ptr(), None, 0, one.data_ptr(), 0, None, 0, m, n, k, k, _capi.BF16, plan, stream)
    torch.cuda.synchronize()
    return status, out

chosen = _capi.TiledPlan()
assert lib.hfrk_tiled_gemm_plan(m, n, k, ctypes.byref(chosen)) == _capi.SUCCESS and chosen.splits > 1
for i in range(64):
    stream = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(stream)) == 0
    assert call(stream, 2)[0] == _capi.SUCCESS, i
assert hip.hipStreamCreate(ctypes.byref(stream)) == 0
assert call(stream, 2)[0] == _capi.NO_WORKSPACE
status, out = call(stream, 0)
want = call(stream, 1)
assert status == want[0] == _capi.SUCCESS and torch.equal(out, want[1])
"""


def test_a_stream_without_a_workspace_does_not_split_k():
    env = dict(os.environ, PYTHONPATH=os.pathsep.join(p for p in sys.path if p))
    subprocess.run([sys.executable, "-c", _NO_WORKSPACE], check=True, timeout=100, env=env)


def _call(lib, dev, weight, packed, out, base, base_stride, m, n, k, dtype, plan, stream=None):
    from hf_rocm_kernels import _capi
    return lib.hfrk_tiled_gemm(dev[0].data_ptr(), weight.data_ptr(), packed, out.data_ptr(), None if base is None else base.data_ptr(),
                               base_stride, dev[2].data_ptr(), 1, dev[3].data_ptr(), 1, m, n, k, k,
                               _capi.F16 if dtype == torch.float16 else _capi.BF16, ctypes.byref(plan),
                               torch.cuda.current_stream().cuda_stream if stream is None else stream)


# stages of 128 bytes over the splits: 11 -> 6 5; 15 -> 4 4 4 3; 21 -> 3 3 3 3 3 2 2 2 (the last stage of each cut to 16 bytes);
# 22 -> 3 3 3 3 3 3 2 2 in both layouts; 13 -> 3 3 3 2 2
@pytest.mark.parametrize("m,n,k,splits", [(130, 136, 1296, 2), (65, 200, 1808, 4), (70, 136, 2576, 8), (257, 264, 2816, 8), (40, 72, 1664, 5)])
def test_uneven_splits_match_the_oracle(m, n, k, splits):
    from hf_rocm_kernels import _capi
    from hf_rocm_kernels.utils.weight_format import pack_weight
    lib = _capi.load()
    a, w, sa, sw = _operands(m, n, k, seed=m + n + k)
    base = torch.randn(m, n, generator=torch.Generator().manual_seed(5)).to(torch.bfloat16)
    check = oracle_checker(a, w.t(), sa, sw, torch.bfloat16, base=base)
    dev, dev_base = [t.cuda() for t in (a, w, sa, sw)], base.cuda()
    layouts = [(0, dev[1])] + ([(1, pack_weight(dev[1]).data)] if k % 256 == 0 else [])
    for shape in range(5):
        first = None
        for packed, weight in layouts:
            out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
            _capi.check(_call(lib, dev, weight, packed, out, dev_base, n, m, n, k, torch.bfloat16, _capi.TiledPlan(shape, splits, 1)), "tiled")
            if first is None:
                check(out)
                first = out
            assert torch.equal(out, first), (shape, packed)


@pytest.mark.parametrize("shape", range(5))
def test_rows_that_are_not_16_byte_aligned(shape):
    """n % 8 == 0, but D and the addend start one element past an aligned address: the element-wise epilogue."""
    from hf_rocm_kernels import _capi
    lib = _capi.load()
    m, n, k = 70, 136, 256
    a, w, sa, sw = _operands(m, n, k, seed=2)
    dev = [t.cuda() for t in (a, w, sa, sw)]
    for rows in (m, 1):
        base = torch.randn(rows * n + 1, device="cuda").to(torch.float16)[1:].view(rows, n)
        for d_off, b in ((1, None), (0, base), (1, base)):
            store = torch.full((m * n + 2,), 7.0, dtype=torch.float16, device="cuda")
            out = store[d_off:d_off + m * n].view(m, n)
            stride = 0 if b is None or rows == 1 else n
            _capi.check(_call(lib, dev, dev[1], 0, out, b, stride, m, n, k, torch.float16, _capi.TiledPlan(shape, 1, 1)), "tiled")
            oracle_checker(a, w.t(), sa, sw, torch.float16, base=None if b is None else b.expand(m, n).contiguous())(out)
            assert (store[:d_off] == 7).all() and (store[d_off + m * n:] == 7).all()


def _split_problem(seed):
    m, n, k = 130, 520, 4096
    a, w, sa, sw = _operands(m, n, k, seed=seed)
    return m, n, k, [t.cuda() for t in (a, w, sa, sw)]


def test_two_streams_with_split_plans_at_once():
    from hf_rocm_kernels import _capi
    lib = _capi.load()
    problems, streams = [_split_problem(s) for s in (1, 2)], [torch.cuda.Stream() for _ in range(2)]
    plan = _capi.TiledPlan(4, 6, 1)
    wants = []
    for m, n, k, dev in problems:
        want = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
        _capi.check(_call(lib, dev, dev[1], 0, want, None, 0, m, n, k, torch.bfloat16, plan), "tiled")
        wants.append(want)
    torch.cuda.synchronize()
    outs = [[], []]
    for _ in range(20):
        for i, (m, n, k, dev) in enumerate(problems):
            with torch.cuda.stream(streams[i]):
                out = torch.zeros(m, n, dtype=torch.bfloat16, device="cuda")
            _capi.check(_call(lib, dev, dev[1], 0, out, None, 0, m, n, k, torch.bfloat16, plan, streams[i].cuda_stream), "tiled")
            outs[i].append(out)
    torch.cuda.synchronize()
    for want, got in zip(wants, outs):
        assert all(torch.equal(g, want) for g in got)


def test_a_captured_split_plan_replays_like_the_eager_call():
    from hf_rocm_kernels import _capi
    lib = _capi.load()
    m, n, k, dev = _split_problem(3)
    plan, stream = _capi.TiledPlan(4, 6, 1), torch.cuda.Stream()
    out = torch.zeros(m, n, dtype=torch.bfloat16, device="cuda")
    torch.cuda.synchronize()

    def call():
        _capi.check(_call(lib, dev, dev[1], 0, out, None, 0, m, n, k, torch.bfloat16, plan, stream.cuda_stream), "tiled")

    with torch.cuda.stream(stream):
        call()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            call()
        for turn in range(5):
            dev[0].copy_(dev[0].flip(0))  # other inputs for every replay
            call()
            torch.cuda.synchronize()
            want = out.clone()
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want) and want.float().abs().sum() > 0, turn


def test_nan_and_infinities_reach_their_rows_and_columns_only():
    from hf_rocm_kernels import _capi
    lib = _capi.load()
    m, n, k = 130, 136, 656
    a, w, sa, sw = _operands(m, n, k, seed=9)
    base = torch.randn(m, n, generator=torch.Generator().manual_seed(5))
    a.view(torch.uint8)[63, k - 1] = 0x7F  # NaN at the end of a row, and of the last, cut stage
    w.view(torch.uint8)[n - 1, 0] = 0xFF
    sa[5], sw[3] = float("inf"), float("nan")
    base[64, 7], base[129, 135 - 1] = float("inf"), float("-inf")
    base = base.to(torch.bfloat16)
    scales = sa.double()[:, None] * sw.double()[None]
    want = (a.double() @ w.double().t()) * scales + base.double()
    slack = want.abs() * 2.0 ** -8 + (a.double().abs() @ w.double().abs().t()) * scales * 2.0 ** -16 + 2.0 ** -126
    dev, dev_base = [t.cuda() for t in (a, w, sa, sw)], base.cuda()
    for shape in range(5):
        for splits in (1, 3):
            out = torch.zeros(m, n, dtype=torch.bfloat16, device="cuda")
            _capi.check(_call(lib, dev, dev[1], 0, out, dev_base, n, m, n, k, torch.bfloat16, _capi.TiledPlan(shape, splits, 1)), "tiled")
            got = out.cpu().double()
            assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf()), (shape, splits)
            fine = want.isfinite()
            assert torch.equal(got[want.isinf()], want[want.isinf()]) and ((got - want).abs() <= slack)[fine].all(), (shape, splits)


@pytest.mark.parametrize("m,n,k", [(65, 264, 4096), (130, 4104, 2304), (201, 1032, 1040), (300, 520, 14336)])
def test_linear_layers_under_the_librarys_plan_match_the_oracle(m, n, k):
    from hf_rocm_kernels.layers import apply_fp8_linear
    from hf_rocm_kernels.utils.weight_format import pack_weight
    a, w, sa, sw = _operands(m, n, k, seed=m + n)
    g = torch.Generator().manual_seed(1)
    bias, residual = torch.randn(n, generator=g).to(torch.bfloat16), torch.randn(m, n, generator=g).to(torch.bfloat16)
    dev = [t.cuda() for t in (a, w, sa, sw)]
    for add, base in ((dict(), None), (dict(bias=bias.cuda()), bias.expand(m, n).contiguous()), (dict(residual=residual.cuda()), residual)):
        check = oracle_checker(a, w.t(), sa, sw, torch.bfloat16, base=base)
        for weight in [dev[1]] + ([pack_weight(dev[1])] if k % 256 == 0 else []):
            check(apply_fp8_linear(dev[0], weight, dev[3], dev[2], **add))


# A process of its own: every stream takes a workspace.
_NEW_STREAMS = """
import ctypes, torch
from hf_rocm_kernels import _capi
lib = _capi.load()
torch.manual_seed(0)
m, n, k = 130, 520, 4096
a, w = (torch.randn(r, k, device="cuda").to(torch.float8_e4m3fn) for r in (m, n))
one = torch.full((1,), 1e-2, device="cuda")
hip = ctypes.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line))

def tiled(out, stream):
    plan = ctypes.byref(_capi.TiledPlan(4, 6, 1))
    return lib.hfrk_tiled_gemm(a.data_ptr(), w.data_ptr(), 0, out.data_ptr(), None, 0, one.data_ptr(), 0, None, 0, m, n, k, k, _capi.BF16, plan, stream)

def skinny(out, stream):  # 64 columns: k is split between workgroups
    return lib.hfrk_skinny_gemm_fused(a.data_ptr(), w.data_ptr(), out.data_ptr(), None, one.data_ptr(), 0, None, 0, None, 64, 64, k, k, _capi.BF16, 0, None, stream)

def outputs():
    return [torch.full((m, n), 7.0, dtype=torch.bfloat16, device="cuda"), torch.full((64, 64), 7.0, dtype=torch.bfloat16, device="cuda")]

want = outputs()
assert tiled(want[0], None) == skinny(want[1], None) == _capi.SUCCESS
for i in range(24):
    stream, got = ctypes.c_void_p(), [outputs() for _ in range(20)]
    assert hip.hipStreamCreateWithFlags(ctypes.byref(stream), 1) == 0  # 1: does not wait for the null stream
    torch.cuda.synchronize()
    torch.cuda._sleep(200000)  # the null stream is busy for about 0.1 ms when the workspace is made, so that clearing ends between launches
    for pair in got:
        assert tiled(pair[0], stream) == skinny(pair[1], stream) == _capi.SUCCESS
    torch.cuda.synchronize()
    for turn, pair in enumerate(got):
        assert all(torch.equal(g, x) for g, x in zip(pair, want)), (i, turn)
"""


def test_the_first_calls_on_a_new_stream():
    env = dict(os.environ, PYTHONPATH=os.pathsep.join(p for p in sys.path if p))
    subprocess.run([sys.executable, "-c", _NEW_STREAMS], check=True, timeout=100, env=env)
