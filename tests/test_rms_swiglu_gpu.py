"""GPU parity of residual-RMSNorm, SwiGLU and the MLP chain against the CPU oracle, with the reference's own test
matrices and criteria (tests/test_residual_rms.py:49-84, tests/test_swiglu.py:23-40) plus bfloat16 and fixtures."""
import glob
import os

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(__file__), "golden")


# The reference's row counts (tests/test_residual_rms.py:49, tests/test_swiglu.py:23), each in its dtype (float16); bfloat16 on
# a subset of them.
def _rows_and_dtypes(rows, bf16_rows):
    return [(r, dt) for r in rows for dt in ([torch.float16, torch.bfloat16] if r in bf16_rows else [torch.float16])]


@pytest.mark.parametrize("force_scalar", [False, True])
@pytest.mark.parametrize("out_fp8,buffer_cols", [(False, 0), (True, 0), (True, 32), (True, 1024)])
@pytest.mark.parametrize("cols", [8, 24, 128, 512, 4096, 16384])
@pytest.mark.parametrize("rows,io_dtype", _rows_and_dtypes([1, 2, 3, 4, 8, 16, 32, 64, 128, 256], (1, 3, 8, 32, 256)))
def test_residual_rms(rows, cols, out_fp8, buffer_cols, io_dtype, force_scalar):
    from hf_rocm_kernels import residual_rms
    from hf_rocm_kernels.operators.residual_rms import generate_residual_rms_data
    from hf_rocm_kernels.utils.testing import compare_x_and_ref_to_precise
    from oracle import residual_rms as orr
    dtype = torch.float8_e4m3fn if out_fp8 else io_dtype
    x, r, w, eps, scale, nb = generate_residual_rms_data(rows, cols, buffer_cols, dtype=dtype, seed=0, io_dtype=io_dtype)
    out, res = residual_rms(x.clone(), r.clone(), w, eps, scale_tensor=scale, next_buffer=nb, force_scalar=force_scalar)
    sc = None if scale is None else scale.cpu()
    ref, ref_res, _ = orr.reference_residual_rms(x.cpu(), r.cpu(), w.cpu(), eps, sc)
    precise, _ = orr.precise_residual_rms(x.cpu(), r.cpu(), w.cpu(), eps, sc)
    # hard checks of the reference's test: zeroed buffer, bit-exact residual
    if nb is not None:
        assert nb.float().abs().sum() == 0
    assert torch.equal(res.cpu().view(torch.int16), ref_res.view(torch.int16))
    assert out.dtype == (torch.float8_e4m3fn if out_fp8 else io_dtype)
    if not out_fp8:
        # 16-bit output follows the reference's rounding points up to the fp32 reduction order of the variance:
        # the normalised value may land one unit in the last place away, and that unit, carried through the
        # multiply by the weight and its rounding, shows as at most two units of the result, on few elements
        from oracle.skinny_gemm import ulp16
        d = (out.cpu().float() - ref.float()).abs().double()
        assert (d <= 2 * ulp16(ref.float(), io_dtype)).all() and (d > 0).float().mean() < 0.02
    dx_max, dr_max, dx_mean, dr_mean, worse_pct, worse_max, worse_mean = compare_x_and_ref_to_precise(
        out.cpu().float(), ref.float(), precise.float())
    # the reference's criteria: no farther from the float64 result than the torch 16-bit path is.  They are
    # statistical (a single fp8 boundary flip is 0.06-0.125 of error), so they are applied where the tensor is
    # large enough for rates to mean something.  The reference's float64 result also does not round the sum to
    # 16 bits, which the kernel and the torch path both do; with bfloat16 that shared 2^-9 error moves fp8
    # rounding boundaries for both, so element-wise "never worse" is only asked of float16.
    assert worse_max <= max(0.25, float(precise.float().abs().max()) * 2.0 ** -3)   # 0.25 in the reference: one fp8 step of its data
    if rows * cols >= 32768:
        assert dx_mean <= dr_mean + 1e-5
        if io_dtype == torch.float16:
            # (fp8 output: the largest error of either path is one rounding-boundary flip, whose size is the fp8 step at the
            # element it happens to hit -- 0.25 below 4, 0.5 from 4 on -- so up to two isolated flips above the torch path's
            # largest are accepted here; the check against the specified result below bounds each by its own step)
            flips = int(((out.cpu().float() - precise.float()).abs() > dr_max).sum())
            assert dx_max <= dr_max or dx_max <= 2.0 ** -9 or (out_fp8 and flips <= 2), (dx_max, dr_max, flips)
            assert worse_pct < (0.1 if out_fp8 else 2.0) and worse_mean < 1e-4
    if out_fp8:
        # what the kernel is specified to compute: exact arithmetic on the rounded sum, one rounding to fp8.
        # fp32 evaluation can only flip values sitting on an fp8 rounding boundary: rare, and one step
        zeros = torch.zeros_like(ref_res)
        spec, _ = orr.precise_residual_rms(ref_res, zeros, w.cpu(), eps, sc)
        d = (out.cpu().float() - spec.float()).abs()
        step = torch.maximum(spec.float().abs() * 2.0 ** -3, torch.tensor(2.0 ** -9))
        assert (d <= step).all()
        assert int((d > 0).sum()) <= max(1, int(2e-4 * d.numel())), int((d > 0).sum())


@pytest.mark.parametrize("force_scalar", [True, False])
@pytest.mark.parametrize("buffer_cols", [0, 1024, 16384])
@pytest.mark.parametrize("hidden_dim", [8, 24, 128, 512, 4096, 6656, 14336])
@pytest.mark.parametrize("rows,io_dtype", _rows_and_dtypes([1, 2, 3, 4, 8, 16, 32, 64, 128, 256, 2048], (1, 3, 8, 32, 256, 2048)))
def test_swiglu(rows, hidden_dim, buffer_cols, io_dtype, force_scalar):
    from hf_rocm_kernels import swiglu
    from hf_rocm_kernels.operators.swiglu import generate_swiglu_data
    from hf_rocm_kernels.utils.testing import compare_x_with_ref
    from oracle import swiglu as osw
    if rows * hidden_dim > 2048 * 6656:
        pytest.skip("larger than the reference's largest case")
    gu, scale, nb = generate_swiglu_data(rows, hidden_dim, buffer_cols, seed=0, io_dtype=io_dtype)
    out = swiglu(gu, scale, nb, force_scalar=force_scalar)
    if nb is not None:
        assert nb.float().abs().sum() == 0
    ref = osw.reference_swiglu(gu.cpu(), scale.cpu())
    assert out.dtype == torch.float8_e4m3fn and out.shape == (rows, hidden_dim)
    # differences can only be fp8 rounding-boundary flips caused by the last bit of the fp32 sigmoid: one fp8 step,
    # and rare (the reference allows < 10 per tensor; here the tensors are also larger, so a rate is used as well)
    o, rf = out.cpu().float(), ref.float()
    d = (o - rf).abs()
    step = torch.maximum(rf.abs() * 2.0 ** -3, torch.tensor(2.0 ** -9))
    assert (d <= step).all()
    changed = int((d > 0).sum())
    assert changed < 10 or changed / d.numel() < 2e-4, changed
    max_err, max_rel, _ = compare_x_with_ref(o * float(scale), rf * float(scale))
    if hidden_dim * rows <= 256 * 6656:
        assert max_rel < 0.15 or max_err < 1e-2


def test_fixtures():
    from hf_rocm_kernels import residual_rms, swiglu
    for f in sorted(glob.glob(os.path.join(GOLDEN, "rms_*.npz"))):
        z = np.load(f)
        dtype = torch.bfloat16 if "bf16" in f else torch.float16
        x = torch.from_numpy(z["input_bits"]).view(dtype).cuda()
        r = torch.from_numpy(z["residual_bits"]).view(dtype).cuda()
        w = torch.from_numpy(z["weight_bits"]).view(dtype).cuda()
        scale = torch.from_numpy(z["scale"]).cuda()
        q, res = residual_rms(x.clone(), r.clone(), w, float(z["eps"]), scale_tensor=scale)
        assert np.array_equal(res.cpu().view(torch.int16).numpy(), z["new_residual_bits"]), f
        d = (q.cpu().float() - torch.from_numpy(z["out_fp8"]).view(torch.float8_e4m3fn).float()).abs()
        assert (d > 0).float().mean() < 0.05 and (d <= q.cpu().float().abs() * 2.0 ** -3 + 2.0 ** -9).all(), f
        h, _ = residual_rms(x.clone(), r.clone(), w, float(z["eps"]))
        hb = torch.from_numpy(z["out16_bits"]).view(dtype)
        assert ((h.cpu().float() - hb.float()).abs() <= hb.float().abs() * 2.0 ** -7).all(), f
    for f in sorted(glob.glob(os.path.join(GOLDEN, "swiglu_*.npz"))):
        z = np.load(f)
        dtype = torch.bfloat16 if "bf16" in f else torch.float16
        gu = torch.from_numpy(z["gate_up_bits"]).view(dtype).cuda()
        q = swiglu(gu, torch.from_numpy(z["scale"]).cuda())
        assert (q.cpu().view(torch.uint8).numpy() != z["out_fp8"]).mean() < 0.01, f


def test_rms_rejects_bad_epsilon_and_mixed_dtypes():
    from hf_rocm_kernels import residual_rms
    x = torch.zeros(4, 64, dtype=torch.float16).cuda()
    w = torch.ones(64, dtype=torch.float16).cuda()
    with pytest.raises(AssertionError, match="epsilon"):
        residual_rms(x, x.clone(), w, 0.0)
    with pytest.raises(AssertionError):
        residual_rms(x, x.clone(), w.to(torch.bfloat16), 1e-5)


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("add_residual", [False, True])
@pytest.mark.parametrize("m", [1, 8, 16])
def test_llama_mlp_chain(m, add_residual, fused):
    """The Llama-3-8B MLP block: hidden 4096, gate_up 28672x4096, down 4096x14336, eps 1e-5, weight ~ 1+N(0,0.1), bf16."""
    from hf_rocm_kernels.combined_ops.llama_mlp import llama_mlp_combined_ops
    from hf_rocm_kernels.utils.fp8 import amax_scale, fp8_quantize
    from oracle import llama_mlp as omlp
    hidden, inter = 4096, 14336
    g = torch.Generator().manual_seed(20 + m)
    dtype = torch.bfloat16
    attn = torch.randn(m, hidden, generator=g).to(dtype)
    resid = torch.randn(m, hidden, generator=g).to(dtype)
    rms_w = (1 + 0.1 * torch.randn(hidden, generator=g)).to(dtype)
    wgu = torch.randn(2 * inter, hidden, generator=g) * 0.02
    wd = torch.randn(hidden, inter, generator=g) * 0.02
    s_gu, s_d = amax_scale(wgu), amax_scale(wd)
    wgu8, wd8 = fp8_quantize(wgu, s_gu)[0], fp8_quantize(wd, s_d)[0]
    in_gu = torch.tensor([6.0 / 448], dtype=torch.float32)    # static activation scales
    in_d = torch.tensor([4.0 / 448], dtype=torch.float32)
    args_cpu = (attn, resid, rms_w, 1e-5, wgu8.t(), in_gu, (in_gu * s_gu).reshape(1), wd8.t(), in_d, (in_d * s_d).reshape(1))
    cpu_args = [t.clone() if isinstance(t, torch.Tensor) else t for t in args_cpu]
    ref_out, ref_res = omlp.reference_llama_mlp(*cpu_args, add_residual=add_residual, exact_norm=True)
    loose_out, _ = omlp.reference_llama_mlp(*cpu_args, add_residual=add_residual, exact_norm=False)
    dev = [t.cuda() if isinstance(t, torch.Tensor) else t for t in args_cpu]
    dev[4], dev[7] = wgu8.cuda().t(), wd8.cuda().t()
    out, res = llama_mlp_combined_ops(*dev, add_residual=add_residual, fused=fused)
    assert torch.equal(res.cpu().view(torch.int16), ref_res.view(torch.int16))
    # Against the chain whose normalisation rounds once (what the kernel computes): the chain quantises twice on the
    # way, so a rare fp8 boundary flip upstream moves a down-projection output by more than the single-GEMM bound;
    # the given tolerance (rtol/atol 1e-2 in bf16) holds for nearly all elements and the rest stay within a few of it.
    o, rf = out.cpu().float(), ref_out.float()
    d = (o - rf).abs()
    tol = 1e-2 + 1e-2 * rf.abs()
    assert (d > tol).float().mean() < 5e-3, float((d > tol).float().mean())
    assert (d <= 4 * tol).all(), float((d / tol).max())
    # Against the reference's torch chain (16-bit roundings inside the normalisation flip ~5% of its fp8 values):
    # agreement at the level those flips allow, a few percent of the output's spread
    dl = (o - loose_out.float()).abs()
    assert float(dl.mean()) < 0.03 * float(loose_out.float().std()) + 1e-2


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("add_residual", [False, True])
@pytest.mark.parametrize("m", [1, 8, 16])
def test_llama_mlp_chain_stage_by_stage(m, add_residual, fused):
    """The Llama-3-8B MLP block held to the strict bar, one stage at a time: every stage of the device chain is compared with the
    oracle's next stage fed with the device's own output of the stage before (so that an fp8 boundary flip upstream cannot
    move the comparison), and the block's result must be, bit for bit, what these stages give when run one by one.
    Order of the chain: hf_rocm_kernels/combined_ops/llama_mlp.py:23-59 of the reference."""
    from hf_rocm_kernels import residual_rms, skinny_gemm, skinny_gemm_add, skinny_gemm_scaled, skinny_gemm_swiglu, swiglu
    from hf_rocm_kernels.combined_ops.llama_mlp import llama_mlp_combined_ops
    from hf_rocm_kernels.utils.fp8 import amax_scale, fp8_quantize
    from oracle import residual_rms as orms
    from oracle import swiglu as osw
    from test_gemm_gpu import _swiglu_oracle, check_against_oracle
    hidden, inter = 4096, 14336
    g = torch.Generator().manual_seed(20 + m)
    dtype = torch.bfloat16
    attn = torch.randn(m, hidden, generator=g).to(dtype)
    resid = torch.randn(m, hidden, generator=g).to(dtype)
    rms_w = (1 + 0.1 * torch.randn(hidden, generator=g)).to(dtype)
    wgu = torch.randn(2 * inter, hidden, generator=g) * 0.02
    wd = torch.randn(hidden, inter, generator=g) * 0.02
    s_gu, s_d = amax_scale(wgu), amax_scale(wd)
    wgu8, wd8 = fp8_quantize(wgu, s_gu)[0].cuda().t(), fp8_quantize(wd, s_d)[0].cuda().t()
    in_gu = torch.tensor([6.0 / 448], dtype=torch.float32).cuda()
    in_d = torch.tensor([4.0 / 448], dtype=torch.float32).cuda()
    out_gu, out_d = (in_gu * s_gu.cuda()).reshape(1), (in_d * s_d.cuda()).reshape(1)
    one = torch.ones(1).cuda()
    block_out, block_res = llama_mlp_combined_ops(attn.cuda(), resid.cuda(), rms_w.cuda(), 1e-5, wgu8, in_gu, out_gu, wd8, in_d, out_d,
                                                  add_residual=add_residual, fused=fused)

    # 1. residual RMSNorm -> fp8: the residual bit for bit, the fp8 values within one step of the float64 result, rarely off
    normalized, res = residual_rms(attn.cuda(), resid.cuda(), rms_w.cuda(), 1e-5, scale_tensor=in_gu)
    want_res = (attn.float() + resid.float()).to(dtype)
    assert torch.equal(res.cpu().view(torch.int16), want_res.view(torch.int16)) and torch.equal(res, block_res)
    q_ref, _ = orms.precise_residual_rms(want_res, torch.zeros_like(want_res), rms_w, 1e-5, in_gu.cpu())
    d = (normalized.cpu().float() - q_ref.float()).abs()
    assert (d <= torch.maximum(q_ref.float().abs() * 2.0 ** -3, torch.tensor(2.0 ** -9))).all() and (d > 0).float().mean() < 0.01

    # 2 + 3. gate_up projection and SwiGLU of the device's own normalised activations
    if fused:
        act = skinny_gemm_swiglu(normalized, wgu8, out_gu, None, in_d, intermediate_dtype=dtype)
        ref, tol = _swiglu_oracle(normalized, wgu8, out_gu, one, in_d, dtype)
        d = (act.cpu().float() - ref.float()).abs()
        assert (d <= tol).all() and (d > 0).float().mean() < 0.02
    else:
        gate_up = skinny_gemm(normalized, wgu8, out_gu, torch.zeros((m, 2 * inter), dtype=dtype, device="cuda"))
        check_against_oracle(gate_up, normalized, wgu8, out_gu, one)      # exact-product bound and rtol/atol 1e-2, every element
        act = swiglu(gate_up, in_d)
        ref = osw.reference_swiglu(gate_up.cpu(), in_d.cpu())
        d = (act.cpu().float() - ref.float()).abs()
        assert (d <= torch.maximum(ref.float().abs() * 2.0 ** -3, torch.tensor(2.0 ** -9))).all() and (d > 0).float().mean() < 0.01

    # 4. down projection (+ residual) of the device's own fp8 activations: every element within the bound and rtol/atol 1e-2
    if add_residual:
        out = skinny_gemm_add(act, wd8, out_d, None, base=res)
    else:
        out = skinny_gemm_scaled(act, wd8, out_d, one)
    check_against_oracle(out, act, wd8, out_d, one, base=res if add_residual else None)
    assert torch.equal(out, block_out), "the block is not the chain of its stages"


# ---- per-row dynamic quantisation ----------------------------------------------------------------------------------------

def _check_dynamic(q_dev, scales_dev, q_ref, scales_ref, y):
    s_dev, s_ref = scales_dev.cpu().double(), scales_ref.double()
    assert ((s_dev - s_ref).abs() <= 4e-6 * s_ref).all(), float(((s_dev - s_ref).abs() / s_ref).max())
    qd = q_dev.cpu().float()
    assert not qd.isnan().any()
    nonzero = y.abs().amax(dim=1) > 0
    assert (qd.abs().amax(dim=1)[nonzero] == 448.0).all()
    d = (qd - q_ref.float()).abs()
    step = torch.maximum(q_ref.float().abs() * 2.0 ** -3, torch.tensor(2.0 ** -9))
    assert (d <= step).all()
    assert (d > 0).float().mean() < 0.01, float((d > 0).float().mean())
    # in real units: dequantised values reproduce y to half an fp8 step (plus the fp32 evaluation of y itself)
    deq = q_dev.cpu().double() * s_dev[:, None]
    assert ((deq - y).abs() <= y.abs() * (2.0 ** -4 + 1e-5) + s_dev[:, None] * 2.0 ** -10 * 1.001).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,cols", [(1, 4096), (8, 4096), (16, 8192), (5, 1024), (3, 32768), (7, 64), (64, 14336)])
def test_residual_rms_dynamic(rows, cols, dtype):
    from hf_rocm_kernels import residual_rms_dynamic
    from oracle import residual_rms as orms
    g = torch.Generator().manual_seed(rows * 100 + cols)
    x = torch.randn(rows, cols, generator=g).to(dtype)
    r = torch.randn(rows, cols, generator=g).to(dtype)
    w = (1 + 0.1 * torch.randn(cols, generator=g)).to(dtype)
    if rows > 2:
        x[1] *= 25.0
    q_ref, z_ref, s_ref, y = orms.precise_residual_rms_dynamic(x, r, w, 1e-5)
    nb = torch.full((rows, 24), 7.0, dtype=dtype).cuda()
    q, res, scales = residual_rms_dynamic(x.cuda(), r.cuda(), w.cuda(), 1e-5, next_buffer=nb)
    assert torch.equal(res.cpu().view(torch.int16), z_ref.view(torch.int16))
    assert (nb == 0).all()
    _check_dynamic(q, scales, q_ref, s_ref, y)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,cols", [(1, 14336), (8, 14336), (16, 28672), (5, 256), (3, 32768), (7, 8)])
def test_swiglu_dynamic(rows, cols, dtype):
    from hf_rocm_kernels import swiglu_dynamic
    from oracle import swiglu as osw
    g = torch.Generator().manual_seed(rows * 100 + cols + 1)
    gu = torch.randn(rows, 2 * cols, generator=g).mul(2.5).to(dtype)
    q_ref, s_ref, y = osw.precise_swiglu_dynamic(gu)
    q, scales = swiglu_dynamic(gu.cuda())
    _check_dynamic(q, scales, q_ref, s_ref, y)


def test_nan_inputs_quantise_like_the_reference_clamp():
    """A NaN does not survive the device's clamp to +-448 (a median of three returns the smaller of the two bounds): it
    is stored as -448 (0xFE), as the reference's clamp stores it, not as the 0x7F the CPU oracle's encoder writes.  The
    dynamic quantiser's row maximum ignores NaN, so the row's scale stays finite and its other values keep their codes."""
    from hf_rocm_kernels import swiglu, swiglu_dynamic
    from oracle import swiglu as osw
    g = torch.Generator().manual_seed(11)
    gu = torch.randn(3, 64, generator=g).to(torch.bfloat16)
    gu[1, 5] = float("nan")        # a gate value
    gu[2, 32 + 9] = float("nan")   # an up value
    scale = torch.tensor([0.05])
    for force_scalar in (False, True):
        out = swiglu(gu.cuda(), scale.cuda(), None, force_scalar=force_scalar).cpu().view(torch.uint8)
        assert out[1, 5] == 0xFE and out[2, 9] == 0xFE
        clean = gu.clone()
        clean[1, 5] = clean[2, 32 + 9] = 0.0
        ref = osw.reference_swiglu(clean, scale).view(torch.uint8)
        mask = torch.ones(3, 32, dtype=torch.bool)
        mask[1, 5] = mask[2, 9] = False
        assert (out[mask].int() - ref[mask].int()).abs().max() <= 1
    q, scales = swiglu_dynamic(gu.cuda())
    assert torch.isfinite(scales).all()
    q = q.cpu().view(torch.uint8)
    assert q[1, 5] == 0xFE and q[2, 9] == 0xFE
    q_ref, s_ref, _ = osw.precise_swiglu_dynamic(clean)
    assert torch.allclose(scales.cpu().reshape(-1), s_ref.reshape(-1).float(), rtol=1e-5)
    assert (q[mask].int() - q_ref.view(torch.uint8)[mask].int()).abs().max() <= 1


def test_dynamic_scales_feed_the_gemm():
    """rms_dynamic -> per-token GEMM: the device's own fp8 rows and scales through the GEMM oracle."""
    from hf_rocm_kernels import residual_rms_dynamic, skinny_gemm_scaled
    from hf_rocm_kernels.utils.fp8 import amax_scale, fp8_quantize
    from oracle import skinny_gemm as og
    g = torch.Generator().manual_seed(11)
    m, hidden, n = 8, 4096, 1024
    x = torch.randn(m, hidden, generator=g).to(torch.bfloat16)
    x[3] *= 40.0
    r = torch.randn(m, hidden, generator=g).to(torch.bfloat16)
    w = (1 + 0.1 * torch.randn(hidden, generator=g)).to(torch.bfloat16)
    wt = torch.randn(n, hidden, generator=g) * 0.02
    sw = amax_scale(wt, dim=1)
    w8 = fp8_quantize(wt, sw)[0]
    q, _, scales = residual_rms_dynamic(x.cuda(), r.cuda(), w.cuda(), 1e-5)
    out = skinny_gemm_scaled(q, w8.cuda().t(), scales, sw.reshape(-1).cuda())
    ref = og.reference_skinny_gemm(q.cpu(), w8.t(), scales.cpu(), sw.reshape(-1), out_dtype=torch.bfloat16)
    assert torch.allclose(out.cpu().float(), ref.float(), rtol=1e-2, atol=1e-2)


def test_dynamic_ops_reject_rows_they_cannot_hold():
    from hf_rocm_kernels import _capi
    lib = _capi.load()
    x = torch.zeros(2, 40000, dtype=torch.bfloat16).cuda()
    q = torch.zeros(2, 40000, dtype=torch.uint8).cuda()
    s = torch.zeros(2).cuda()
    w = torch.zeros(40000, dtype=torch.bfloat16).cuda()
    rms = lambda cols: lib.hfrk_residual_rms_dynamic(x.data_ptr(), x.data_ptr(), w.data_ptr(), 1e-5, q.data_ptr(), s.data_ptr(),
                                                     None, 2, cols, 0, _capi.BF16, None)
    assert rms(36) == _capi.BAD_SHAPE          # cols % 8 != 0
    assert rms(40000) == _capi.BAD_SHAPE       # wider than the register cache
    assert lib.hfrk_swiglu_dynamic(x.data_ptr(), q.data_ptr(), s.data_ptr(), None, 1, 20004, 0, _capi.BF16, None) == _capi.BAD_SHAPE
    assert lib.hfrk_swiglu_dynamic(x.data_ptr() + 2, q.data_ptr(), s.data_ptr(), None, 1, 64, 0, _capi.BF16, None) == _capi.BAD_ALIGNMENT


@pytest.mark.parametrize("packed", [False, True])
def test_captured_mlp_block_replays_like_the_eager_block(packed, monkeypatch):
    """LlamaMlpGraph: the fused block as one graph launch.  Replayed several times with fresh inputs, with the
    program's own eager launches and synchronisations in between; every replay, and every call of the object, must equal the launches of the
    wrappers (without the native block) bit for bit."""
    import sys
    from hf_rocm_kernels.combined_ops.llama_mlp import LlamaMlpGraph, llama_mlp_combined_ops
    module = sys.modules["hf_rocm_kernels.combined_ops.llama_mlp"]
    from hf_rocm_kernels.utils.fp8 import amax_scale, fp8_quantize
    from hf_rocm_kernels.utils.weight_format import pack_weight
    g = torch.Generator().manual_seed(5)
    m, hidden, inter = 8, 1024, 2816
    wn = (1 + 0.1 * torch.randn(hidden, generator=g)).to(torch.bfloat16).cuda()
    wgu = (0.02 * torch.randn(2 * inter, hidden, generator=g)).cuda()
    wd = (0.02 * torch.randn(hidden, inter, generator=g)).cuda()
    qgu, sgu = fp8_quantize(wgu, amax_scale(wgu))
    qd, sd = fp8_quantize(wd, amax_scale(wd))
    w_gu = pack_weight(qgu) if packed else qgu.t()
    w_d = pack_weight(qd) if packed else qd.t()
    s_in, s_mid = torch.full((1,), 0.02, device="cuda"), torch.full((1,), 0.01, device="cuda")
    args = (wn, 1e-5, w_gu, s_in, (s_in * sgu).view(1), w_d, s_mid, (s_mid * sd).view(1))
    block = LlamaMlpGraph(m, hidden, *args)
    for step in range(4):
        x = torch.randn(m, hidden, generator=g).to(torch.bfloat16).cuda()
        res = torch.randn(m, hidden, generator=g).to(torch.bfloat16).cuda()
        with monkeypatch.context() as patch:
            patch.setattr(module, "_llama_mlp", lambda *a: False)
            want, want_res = llama_mlp_combined_ops(x, res.clone(), *args, add_residual=True, fused=True)
        torch.cuda.synchronize()
        block.attn_output.copy_(x)
        block.residual.copy_(res)
        block.mlp_output.zero_()
        block.graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(block.mlp_output, want) and torch.equal(block.residual, want_res), step
        block.mlp_output.zero_()
        got, got_res = block(x, res)
        torch.cuda.synchronize()
        assert torch.equal(got, want) and torch.equal(got_res, want_res), step
        assert got.float().abs().sum() > 0


@pytest.mark.gpu
def test_captured_mlp_block_keeps_its_operands_alive():
    """A replay reads the weights and scales by address, so the block must own them: a caller that drops its own references (and a
    cache that is emptied afterwards) must not take them away."""
    import gc
    import weakref
    from hf_rocm_kernels.combined_ops.llama_mlp import LlamaMlpGraph
    from hf_rocm_kernels.utils.weight_format import pack_weight
    hidden, inter = 256, 512
    one = torch.ones(1, device="cuda")
    args = [torch.ones(hidden, dtype=torch.bfloat16, device="cuda"), 1e-5,
            pack_weight(torch.zeros(2 * inter, hidden, device="cuda").to(torch.float8_e4m3fn)), one,
            one.clone(), torch.zeros(hidden, inter, device="cuda").to(torch.float8_e4m3fn).t(), one.clone(), one.clone()]
    refs = [weakref.ref(a) for a in args if not isinstance(a, float)]
    block = LlamaMlpGraph(1, hidden, *args)
    del args, one
    gc.collect()
    assert all(r() is not None for r in refs)
    del block


@pytest.mark.gpu
@pytest.mark.parametrize("fused", [False, True])
def test_traced_mlp_block_equals_the_eager_block(fused):
    """The operators have shape-only implementations, so torch can trace the block as one graph (no graph break) and
    functionalise its in-place writes; the traced function must return what the eager one does, bit for bit."""
    from hf_rocm_kernels.combined_ops.llama_mlp import llama_mlp_combined_ops
    from hf_rocm_kernels.utils.fp8 import amax_scale, fp8_quantize
    g = torch.Generator().manual_seed(6)
    m, hidden, inter = 8, 1024, 2816
    wn = (1 + 0.1 * torch.randn(hidden, generator=g)).to(torch.bfloat16).cuda()
    wgu = (0.02 * torch.randn(2 * inter, hidden, generator=g)).cuda()
    wd = (0.02 * torch.randn(hidden, inter, generator=g)).cuda()
    qgu, sgu = fp8_quantize(wgu, amax_scale(wgu))
    qd, sd = fp8_quantize(wd, amax_scale(wd))
    s_in, s_mid = torch.full((1,), 0.02, device="cuda"), torch.full((1,), 0.01, device="cuda")
    args = (wn, 1e-5, qgu.t(), s_in, (s_in * sgu).view(1), qd.t(), s_mid, (s_mid * sd).view(1))

    def block(x, res):
        return llama_mlp_combined_ops(x, res, *args, add_residual=True, fused=fused)

    traced = torch.compile(block, backend="aot_eager", fullgraph=True)
    for step in range(3):
        x = torch.randn(m, hidden, generator=g).to(torch.bfloat16).cuda()
        res = torch.randn(m, hidden, generator=g).to(torch.bfloat16).cuda()
        want, want_res = block(x, res.clone())
        got, got_res = traced(x, res.clone())
        torch.cuda.synchronize()
        assert torch.equal(got, want) and torch.equal(got_res, want_res), step
        assert got.float().abs().sum() > 0


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("fp8", [True, False])
@pytest.mark.parametrize("rows,cols", [(1792, 16384), (7168, 4096), (3585, 8192)])
def test_large_inputs_give_the_bits_of_their_halves(rows, cols, fp8, dtype):
    """From 28 Mi values on the input is read past the caches; its halves are not.  Rows are independent."""
    from hf_rocm_kernels import residual_rms
    g = torch.Generator(device="cuda").manual_seed(rows)
    x, res = (torch.randn(rows, cols, device="cuda", generator=g).to(dtype) for _ in range(2))
    w = (1 + 0.1 * torch.randn(cols, device="cuda", generator=g)).to(dtype)
    scale = torch.tensor([6.0 / 448], device="cuda") if fp8 else None
    whole, sums = residual_rms(x, res.clone(), w, 1e-5, scale)
    half = rows // 2
    for part in (slice(0, half), slice(half, rows)):
        out, sum_ = residual_rms(x[part], res[part].clone(), w, 1e-5, scale)
        assert torch.equal(whole[part].view(torch.uint8), out.view(torch.uint8)) and torch.equal(sums[part], sum_)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("num_threads", [0, 192, 1024])
@pytest.mark.parametrize("rows,cols", [(4007, 8272), (3909, 8192), (2001, 16384)])
def test_large_swiglu_gives_the_bits_of_its_halves(rows, cols, num_threads, dtype):
    """From 4 million pieces of 8 values on a workgroup's pieces follow one another; those of the halves are a launch apart."""
    from hf_rocm_kernels import swiglu
    g = torch.Generator(device="cuda").manual_seed(rows)
    gate_up = torch.randn(rows, 2 * cols, device="cuda", generator=g).to(dtype)
    scale = torch.tensor([8.0 / 448], device="cuda")
    whole = swiglu(gate_up, scale, num_threads=num_threads)
    half = rows // 2
    for part in (slice(0, half), slice(half, rows)):
        assert torch.equal(whole[part].view(torch.uint8), swiglu(gate_up[part], scale).view(torch.uint8))
