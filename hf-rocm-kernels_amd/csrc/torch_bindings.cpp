// torch.ops._HFRK_C.* -- the operator surface of the reference (csrc/torch_bindings.cpp:20-44, csrc/ops.h:8-19),
// same schemas, implemented by forwarding plain pointers to the C ABI of libhfrk_gfx950.so.
// No kernel lives here: this file only unpacks tensors, checks them, selects device and stream.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/library.h>

#include "hfrk_gfx950.h"

namespace {

// Make the tensor's device current for the duration of a call (the launchers use the current device).
struct DeviceScope {
    c10::DeviceIndex prev;
    bool changed;
    explicit DeviceScope(const at::Tensor& t) : prev(c10::hip::current_device()), changed(false) {
        const c10::DeviceIndex want = t.device().index();
        if (want >= 0 && want != prev) {
            c10::hip::set_device(want);
            changed = true;
        }
    }
    ~DeviceScope() {
        if (changed) c10::hip::set_device(prev);
    }
};

void* current_stream(const at::Tensor& t) {
    return static_cast<void*>(c10::hip::getCurrentHIPStream(t.device().index()).stream());
}

int dtype16(const at::Tensor& t, const char* name) {
    if (t.scalar_type() == at::kBFloat16) return HFRK_BF16;
    if (t.scalar_type() == at::kHalf) return HFRK_F16;
    TORCH_CHECK(false, name, " must be float16 or bfloat16, got ", t.scalar_type());
}

void check_fp8(const at::Tensor& t, const char* name) {
    TORCH_CHECK(t.scalar_type() != at::kFloat8_e4m3fnuz, name,
                " is float8_e4m3fnuz: gfx950 computes in OCP float8_e4m3fn (same bits read as twice the fnuz value); "
                "re-encode the tensor or pass a float8_e4m3fn view and double its scale");
    TORCH_CHECK(t.scalar_type() == at::kFloat8_e4m3fn, name, " must be float8_e4m3fn, got ", t.scalar_type());
}

void check_same_device(const at::Tensor& ref, const at::Tensor& t, const char* name) {
    TORCH_CHECK(t.device() == ref.device(), name, " is on ", t.device(), " but expected ", ref.device());
}

void raise_on(int status, const char* op) {
    TORCH_CHECK(status == HFRK_SUCCESS, op, " failed: ", hfrk_status_string(status), " (status ", status,
                ", hip error ", hfrk_last_hip_error(), ")");
}

// reference: csrc/op_src/increment/increment_op.cu:3
void increment(at::Tensor& x) { x += 1; }

// reference: csrc/op_src/residual_rms/residual_rms_dispatch.cu:8-63
void residual_rms(at::Tensor& input, at::Tensor& residual, at::Tensor& weight, at::Tensor& scale_tensor, double epsilon,
                  at::Tensor& output, at::Tensor& next_buffer, int64_t num_threads, bool force_scalar) {
    TORCH_CHECK(input.dim() == 2 && input.is_contiguous(), "input must be a contiguous [rows, cols] tensor");
    TORCH_CHECK(residual.sizes() == input.sizes() && residual.is_contiguous(), "residual must match input and be contiguous");
    TORCH_CHECK(weight.dim() == 1 && weight.size(0) == input.size(1) && weight.is_contiguous(), "weight must be [cols]");
    TORCH_CHECK(output.sizes() == input.sizes() && output.is_contiguous(), "output must match input and be contiguous");
    const int io = dtype16(input, "input");
    TORCH_CHECK(residual.scalar_type() == input.scalar_type() && weight.scalar_type() == input.scalar_type(),
                "input, residual and weight must share one 16-bit dtype");
    int out = io;
    if (output.scalar_type() != input.scalar_type()) {
        check_fp8(output, "output");
        out = HFRK_FP8_E4M3FN;
        TORCH_CHECK(scale_tensor.numel() == 1 && scale_tensor.scalar_type() == at::kFloat, "fp8 output needs a one-element float32 scale_tensor");
        check_same_device(input, scale_tensor, "scale_tensor");
    }
    check_same_device(input, residual, "residual");
    check_same_device(input, weight, "weight");
    check_same_device(input, output, "output");
    int64_t buffer_cols = 0;
    void* nb = nullptr;
    if (next_buffer.numel() > 0) {
        TORCH_CHECK(next_buffer.dim() == 2 && next_buffer.size(0) == input.size(0) && next_buffer.is_contiguous(),
                    "next_buffer must be a contiguous [rows, buffer_cols] tensor");
        TORCH_CHECK(next_buffer.element_size() == 2, "next_buffer must hold 16-bit elements");
        check_same_device(input, next_buffer, "next_buffer");
        buffer_cols = next_buffer.size(1);
        nb = next_buffer.data_ptr();
    }
    DeviceScope scope(input);
    raise_on(hfrk_residual_rms(input.data_ptr(), residual.data_ptr(), weight.data_ptr(),
                               out == HFRK_FP8_E4M3FN ? scale_tensor.data_ptr<float>() : nullptr, (float)epsilon,
                               output.data_ptr(), nb, (int)input.size(0), (int)input.size(1), (int)buffer_cols, io, out,
                               (int)num_threads, force_scalar ? 1 : 0, current_stream(input)),
             "residual_rms");
}

// reference: csrc/op_src/swiglu/swiglu_dispatch.cu:8-42
void swiglu(at::Tensor& gate_up, at::Tensor& scale_tensor, at::Tensor& output, at::Tensor& next_buffer, int64_t num_threads,
            bool force_scalar) {
    TORCH_CHECK(gate_up.dim() == 2 && gate_up.is_contiguous() && gate_up.size(1) % 2 == 0,
                "gate_up must be a contiguous [rows, 2*cols] tensor");
    const int io = dtype16(gate_up, "gate_up");
    const int64_t rows = gate_up.size(0), cols = gate_up.size(1) / 2;
    check_fp8(output, "output");
    TORCH_CHECK(output.dim() == 2 && output.size(0) == rows && output.size(1) == cols && output.is_contiguous(),
                "output must be a contiguous [rows, cols] tensor");
    TORCH_CHECK(scale_tensor.numel() == 1 && scale_tensor.scalar_type() == at::kFloat, "scale_tensor must be one float32");
    check_same_device(gate_up, scale_tensor, "scale_tensor");
    check_same_device(gate_up, output, "output");
    int64_t buffer_cols = 0;
    void* nb = nullptr;
    if (next_buffer.numel() > 0) {
        TORCH_CHECK(next_buffer.dim() == 2 && next_buffer.size(0) == rows && next_buffer.is_contiguous(),
                    "next_buffer must be a contiguous [rows, buffer_cols] tensor");
        TORCH_CHECK(next_buffer.element_size() == 2, "next_buffer must hold 16-bit elements");
        check_same_device(gate_up, next_buffer, "next_buffer");
        buffer_cols = next_buffer.size(1);
        nb = next_buffer.data_ptr();
    }
    DeviceScope scope(gate_up);
    raise_on(hfrk_swiglu(gate_up.data_ptr(), scale_tensor.data_ptr<float>(), output.data_ptr(), nb, (int)rows, (int)cols,
                         (int)buffer_cols, io, (int)(num_threads < 0 ? 0 : num_threads), force_scalar ? 1 : 0,
                         current_stream(gate_up)),
             "swiglu");
}

// Elements between the weight's rows, which the C ABI takes as an int: cut to one, a larger stride would name other rows.
int row_stride(const at::Tensor& B) {
    TORCH_CHECK(B.size(1) <= 1 || B.stride(1) < (int64_t(1) << 31), "the weight's rows must be less than 2^31 elements apart, got ", B.stride(1));
    return (int)B.stride(1);
}

void check_gemm_operands(const at::Tensor& A, const at::Tensor& B, const at::Tensor& D) {
    TORCH_CHECK(A.dim() == 2 && A.is_contiguous(), "A must be a contiguous [m, k] tensor");
    TORCH_CHECK(B.dim() == 2 && B.size(0) == A.size(1) && B.stride(0) == 1, "B must be [k, n] with unit stride along k");
    TORCH_CHECK(D.dim() == 2 && D.size(0) == A.size(0) && D.size(1) == B.size(1) && D.is_contiguous(),
                "D must be a contiguous [m, n] tensor");
    check_fp8(A, "A");
    check_fp8(B, "B");
    check_same_device(A, B, "B");
    check_same_device(A, D, "D");
}

// reference: csrc/op_src/skinny_gemm/skinny_gemm_binding.cu:16-42.  Returns the status code like the reference;
// misuse of dtypes/devices raises instead of reading garbage.
int64_t skinny_gemm_tb(at::Tensor& A, at::Tensor& B, at::Tensor& D, at::Tensor& scale_tensor, int64_t split_k,
                       int64_t A_producers, int64_t B_producers, int64_t consumers, int64_t a_lanes, int64_t b_lanes,
                       int64_t qsize, int64_t op_m, int64_t ops) {
    check_gemm_operands(A, B, D);
    TORCH_CHECK(scale_tensor.numel() == 1 && scale_tensor.scalar_type() == at::kFloat, "scale_tensor must be one float32");
    check_same_device(A, scale_tensor, "scale_tensor");
    const int d_dtype = dtype16(D, "D");
    DeviceScope scope(A);  // before the stream is looked up
    return hfrk_skinny_gemm(A.data_ptr(), B.data_ptr(), D.data_ptr(), scale_tensor.data_ptr<float>(), (int)A.size(0),
                            (int)B.size(1), (int)A.size(1), row_stride(B), (int)split_k, (int)A_producers,
                            (int)B_producers, (int)consumers, (int)a_lanes, (int)b_lanes, (int)qsize, (int)op_m, (int)ops,
                            d_dtype, current_stream(A));
}

// Per-token (scale_a: 1 or m values) x per-output-channel (scale_b: 1 or n values) scaling.  No reference counterpart.
int64_t skinny_gemm_scaled(at::Tensor& A, at::Tensor& B, at::Tensor& D, at::Tensor& scale_a, at::Tensor& scale_b,
                           bool accumulate) {
    check_gemm_operands(A, B, D);
    const int64_t m = A.size(0), n = B.size(1);
    TORCH_CHECK(scale_a.scalar_type() == at::kFloat && scale_a.is_contiguous() && (scale_a.numel() == 1 || scale_a.numel() == m),
                "scale_a must be float32 with 1 or m elements");
    TORCH_CHECK(scale_b.scalar_type() == at::kFloat && scale_b.is_contiguous() && (scale_b.numel() == 1 || scale_b.numel() == n),
                "scale_b must be float32 with 1 or n elements");
    check_same_device(A, scale_a, "scale_a");
    check_same_device(A, scale_b, "scale_b");
    const int d_dtype = dtype16(D, "D");
    DeviceScope scope(A);
    return hfrk_skinny_gemm_ex(A.data_ptr(), B.data_ptr(), D.data_ptr(), scale_a.data_ptr<float>(),
                               scale_a.numel() == 1 ? 0 : 1, scale_b.data_ptr<float>(), scale_b.numel() == 1 ? 0 : 1, (int)m,
                               (int)n, (int)A.size(1), row_stride(B), d_dtype, accumulate ? 1 : 0, nullptr,
                               current_stream(A));
}

static void next_buffer_args(const at::Tensor& like, const at::Tensor& next_buffer, int64_t rows, void** nb, int64_t* buffer_cols) {
    *nb = nullptr;
    *buffer_cols = 0;
    if (next_buffer.numel() > 0) {
        TORCH_CHECK(next_buffer.dim() == 2 && next_buffer.size(0) == rows && next_buffer.is_contiguous(),
                    "next_buffer must be a contiguous [rows, buffer_cols] tensor");
        TORCH_CHECK(next_buffer.element_size() == 2, "next_buffer must hold 16-bit elements");
        check_same_device(like, next_buffer, "next_buffer");
        *buffer_cols = next_buffer.size(1);
        *nb = next_buffer.data_ptr();
    }
}

// residual RMSNorm with per-row dynamic fp8 quantisation: output fp8 [rows, cols], scales fp32 [rows].  No reference counterpart.
void residual_rms_dynamic(at::Tensor& input, at::Tensor& residual, at::Tensor& weight, double epsilon, at::Tensor& output,
                          at::Tensor& scales, at::Tensor& next_buffer) {
    TORCH_CHECK(input.dim() == 2 && input.is_contiguous(), "input must be a contiguous [rows, cols] tensor");
    TORCH_CHECK(residual.sizes() == input.sizes() && residual.is_contiguous(), "residual must match input and be contiguous");
    TORCH_CHECK(weight.dim() == 1 && weight.size(0) == input.size(1) && weight.is_contiguous(), "weight must be [cols]");
    TORCH_CHECK(output.sizes() == input.sizes() && output.is_contiguous(), "output must match input and be contiguous");
    const int io = dtype16(input, "input");
    TORCH_CHECK(residual.scalar_type() == input.scalar_type() && weight.scalar_type() == input.scalar_type(),
                "input, residual and weight must share one 16-bit dtype");
    check_fp8(output, "output");
    TORCH_CHECK(scales.scalar_type() == at::kFloat && scales.is_contiguous() && scales.numel() == input.size(0),
                "scales must be a contiguous float32 tensor with one element per row");
    check_same_device(input, residual, "residual");
    check_same_device(input, weight, "weight");
    check_same_device(input, output, "output");
    check_same_device(input, scales, "scales");
    void* nb;
    int64_t buffer_cols;
    next_buffer_args(input, next_buffer, input.size(0), &nb, &buffer_cols);
    DeviceScope scope(input);
    raise_on(hfrk_residual_rms_dynamic(input.data_ptr(), residual.data_ptr(), weight.data_ptr(), (float)epsilon, output.data_ptr(),
                                       scales.data_ptr<float>(), nb, (int)input.size(0), (int)input.size(1), (int)buffer_cols, io,
                                       current_stream(input)),
             "residual_rms_dynamic");
}

// SwiGLU with per-row dynamic fp8 quantisation.  No reference counterpart.
void swiglu_dynamic(at::Tensor& gate_up, at::Tensor& output, at::Tensor& scales, at::Tensor& next_buffer) {
    TORCH_CHECK(gate_up.dim() == 2 && gate_up.is_contiguous() && gate_up.size(1) % 2 == 0,
                "gate_up must be a contiguous [rows, 2*cols] tensor");
    const int io = dtype16(gate_up, "gate_up");
    const int64_t rows = gate_up.size(0), cols = gate_up.size(1) / 2;
    check_fp8(output, "output");
    TORCH_CHECK(output.dim() == 2 && output.size(0) == rows && output.size(1) == cols && output.is_contiguous(),
                "output must be a contiguous [rows, cols] tensor");
    TORCH_CHECK(scales.scalar_type() == at::kFloat && scales.is_contiguous() && scales.numel() == rows,
                "scales must be a contiguous float32 tensor with one element per row");
    check_same_device(gate_up, output, "output");
    check_same_device(gate_up, scales, "scales");
    void* nb;
    int64_t buffer_cols;
    next_buffer_args(gate_up, next_buffer, rows, &nb, &buffer_cols);
    DeviceScope scope(gate_up);
    raise_on(hfrk_swiglu_dynamic(gate_up.data_ptr(), output.data_ptr(), scales.data_ptr<float>(), nb, (int)rows, (int)cols,
                                 (int)buffer_cols, io, current_stream(gate_up)),
             "swiglu_dynamic");
}

// 16-bit [rows, cols] -> float8_e4m3fn: with one static scale (the reference's fp8_quantize, hf_rocm_kernels/utils/fp8.py:6-29,
// as one kernel) or, scale_tensor None, one dynamic scale per row written to `scales`.
void quantize_fp8(at::Tensor& input, const std::optional<at::Tensor>& scale_tensor, at::Tensor& output, at::Tensor& scales) {
    TORCH_CHECK(input.dim() == 2 && input.is_contiguous(), "input must be a contiguous [rows, cols] tensor");
    const int io = dtype16(input, "input");
    check_fp8(output, "output");
    TORCH_CHECK(output.sizes() == input.sizes() && output.is_contiguous(), "output must match input and be contiguous");
    check_same_device(input, output, "output");
    const float* static_scale = nullptr;
    float* scales_ptr = nullptr;
    if (scale_tensor.has_value()) {
        TORCH_CHECK(scale_tensor->numel() == 1 && scale_tensor->scalar_type() == at::kFloat, "scale_tensor must be one float32");
        check_same_device(input, *scale_tensor, "scale_tensor");
        static_scale = scale_tensor->data_ptr<float>();
    } else {
        TORCH_CHECK(scales.scalar_type() == at::kFloat && scales.is_contiguous() && scales.numel() == input.size(0),
                    "scales must be a contiguous float32 tensor with one element per row");
        check_same_device(input, scales, "scales");
        scales_ptr = scales.data_ptr<float>();
    }
    DeviceScope scope(input);
    raise_on(hfrk_quantize_fp8(input.data_ptr(), static_scale, output.data_ptr(), scales_ptr, (int)input.size(0), (int)input.size(1), io,
                               current_stream(input)),
             "quantize_fp8");
}

// The GEMM with the surrounding element-wise work folded in.  No reference counterpart as one op.
//   epilogue 0: D = (base ? base : 0) + scale_a x scale_b x A.B, base a 16-bit [m,n] tensor (D itself, a residual) or None
//   epilogue 1: B is a gate_up weight [k, 2*inter]; D fp8 [m, inter] = e4m3fn(silu(gate) * up / out_scale), the two
//               projections rounded to `intermediate_dtype` (0 = float16, 1 = bfloat16) first
// Shared by skinny_gemm_fused (B = the [k, n] view of a row-major weight) and skinny_gemm_packed (B = the buffer
// pack_weight wrote, n given by the caller).
int64_t gemm_fused_common(at::Tensor& A, at::Tensor& B, bool packed, int64_t n, at::Tensor& D,
                          const std::optional<at::Tensor>& base, at::Tensor& scale_a,
                          const std::optional<at::Tensor>& scale_b, const std::optional<at::Tensor>& out_scale,
                          int64_t epilogue, int64_t intermediate_dtype) {
    TORCH_CHECK(A.dim() == 2 && A.is_contiguous(), "A must be a contiguous [m, k] tensor");
    check_fp8(A, "A");
    check_fp8(B, "B");
    if (packed) {
        TORCH_CHECK(n >= 1 && n < (int64_t(1) << 30) && A.size(1) < (int64_t(1) << 30), "n and k must fit 30 bits");
        const size_t plain = hfrk_packed_weight_bytes((int)n, (int)A.size(1)), scaled = hfrk_packed_weight_bytes_scaled((int)n, (int)A.size(1));
        TORCH_CHECK(B.is_contiguous() && B.numel() > 0 && ((size_t)B.numel() == plain || (size_t)B.numel() == scaled),
                    "B must be the packed buffer of a [n, k] weight (pack_weight, pack_weight_scaled) with k = A.size(1)");
    } else {
        TORCH_CHECK(B.dim() == 2 && B.size(0) == A.size(1) && B.stride(0) == 1, "B must be [k, n] with unit stride along k");
    }
    check_same_device(A, B, "B");
    check_same_device(A, D, "D");
    const int64_t m = A.size(0);
    TORCH_CHECK(scale_a.scalar_type() == at::kFloat && scale_a.is_contiguous() && (scale_a.numel() == 1 || scale_a.numel() == m),
                "scale_a must be float32 with 1 or m elements");
    check_same_device(A, scale_a, "scale_a");
    // None = 1, in either weight layout: the scales a pack_weight_scaled buffer carries apply only when the caller passes
    // them (PackedWeight.scales is a view of that part of the buffer), so one call means one thing whatever the layout.
    const float* scale_b_ptr = nullptr;
    int sb_stride = 0;
    if (scale_b.has_value()) {
        TORCH_CHECK(scale_b->scalar_type() == at::kFloat && scale_b->is_contiguous() && (scale_b->numel() == 1 || scale_b->numel() == n),
                    "scale_b must be float32 with 1 or n elements");
        check_same_device(A, *scale_b, "scale_b");
        scale_b_ptr = scale_b->data_ptr<float>();
        sb_stride = scale_b->numel() == 1 ? 0 : 1;
    }
    int d_dtype;
    const void* base_ptr = nullptr;
    const float* out_scale_ptr = nullptr;
    if (epilogue == HFRK_EPILOGUE_SWIGLU) {
        TORCH_CHECK(n % 2 == 0 && D.dim() == 2 && D.size(0) == m && D.size(1) == n / 2 && D.is_contiguous(),
                    "D must be a contiguous [m, n/2] tensor");
        check_fp8(D, "D");
        TORCH_CHECK(out_scale.has_value() && out_scale->numel() == 1 && out_scale->scalar_type() == at::kFloat,
                    "out_scale must be one float32");
        check_same_device(A, *out_scale, "out_scale");
        TORCH_CHECK(!base.has_value(), "base cannot be combined with the SwiGLU epilogue");
        TORCH_CHECK(intermediate_dtype == HFRK_F16 || intermediate_dtype == HFRK_BF16, "intermediate_dtype must be 0 (float16) or 1 (bfloat16)");
        d_dtype = (int)intermediate_dtype;
        out_scale_ptr = out_scale->data_ptr<float>();
    } else {
        TORCH_CHECK(D.dim() == 2 && D.size(0) == m && D.size(1) == n && D.is_contiguous(), "D must be a contiguous [m, n] tensor");
        d_dtype = dtype16(D, "D");
        if (base.has_value()) {
            TORCH_CHECK(base->sizes() == D.sizes() && base->is_contiguous() && base->scalar_type() == D.scalar_type(),
                        "base must be a contiguous tensor with D's shape and dtype");
            check_same_device(A, *base, "base");
            base_ptr = base->data_ptr();
        }
    }
    DeviceScope scope(A);
    if (packed)
        return hfrk_skinny_gemm_packed(A.data_ptr(), B.data_ptr(), D.data_ptr(), base_ptr, scale_a.data_ptr<float>(),
                                       scale_a.numel() == 1 ? 0 : 1, scale_b_ptr, sb_stride, out_scale_ptr, (int)m, (int)n,
                                       (int)A.size(1), d_dtype, (int)epilogue, nullptr, current_stream(A));
    return hfrk_skinny_gemm_fused(A.data_ptr(), B.data_ptr(), D.data_ptr(), base_ptr, scale_a.data_ptr<float>(),
                                  scale_a.numel() == 1 ? 0 : 1, scale_b_ptr, sb_stride, out_scale_ptr, (int)m, (int)n, (int)A.size(1), row_stride(B), d_dtype, (int)epilogue,
                                  nullptr, current_stream(A));
}

int64_t skinny_gemm_fused(at::Tensor& A, at::Tensor& B, at::Tensor& D, const std::optional<at::Tensor>& base,
                          at::Tensor& scale_a, const std::optional<at::Tensor>& scale_b, const std::optional<at::Tensor>& out_scale,
                          int64_t epilogue, int64_t intermediate_dtype) {
    TORCH_CHECK(B.dim() == 2, "B must be [k, n] with unit stride along k");
    return gemm_fused_common(A, B, false, B.size(1), D, base, scale_a, scale_b, out_scale, epilogue, intermediate_dtype);
}

// skinny_gemm_fused with the residual RMSNorm of its activations as the kernel's prologue (no reference counterpart as one
// op: the reference launches residual_rms, then skinny_gemm).  residual_out <- input + residual; the GEMM multiplies
// e4m3fn(rmsnorm(residual_out) * rms_weight / act_scale) by B.  Returns the launcher's status: 7 (HFRK_BAD_SHAPE) where the
// prologue does not exist (more than 8 rows, k other than 4096 / 8192, rows that do not deal out evenly).
int64_t skinny_gemm_rms_fused(at::Tensor& input, at::Tensor& residual, at::Tensor& residual_out, at::Tensor& rms_weight,
                              double epsilon, at::Tensor& act_scale, at::Tensor& B, at::Tensor& D,
                              const std::optional<at::Tensor>& base, at::Tensor& scale_a, const std::optional<at::Tensor>& scale_b,
                              const std::optional<at::Tensor>& out_scale, int64_t epilogue, int64_t intermediate_dtype) {
    TORCH_CHECK(input.dim() == 2 && input.is_contiguous(), "input must be a contiguous [m, k] tensor");
    const int io = dtype16(input, "input");
    const int64_t m = input.size(0), k = input.size(1);
    TORCH_CHECK(residual.sizes() == input.sizes() && residual.is_contiguous() && residual.scalar_type() == input.scalar_type(),
                "residual must be a contiguous tensor with input's shape and dtype");
    TORCH_CHECK(residual_out.sizes() == input.sizes() && residual_out.is_contiguous() && residual_out.scalar_type() == input.scalar_type(),
                "residual_out must be a contiguous tensor with input's shape and dtype");
    TORCH_CHECK(rms_weight.dim() == 1 && rms_weight.size(0) == k && rms_weight.is_contiguous() && rms_weight.scalar_type() == input.scalar_type(),
                "rms_weight must be a contiguous [k] tensor of input's dtype");
    TORCH_CHECK(act_scale.numel() == 1 && act_scale.scalar_type() == at::kFloat, "act_scale must be one float32");
    TORCH_CHECK(scale_a.numel() == 1 && scale_a.scalar_type() == at::kFloat, "scale_a must be one float32");
    check_fp8(B, "B");
    TORCH_CHECK(B.dim() == 2 && B.size(0) == k && B.stride(0) == 1, "B must be [k, n] with unit stride along k");
    const int64_t n = B.size(1);
    for (const at::Tensor* t : {&residual, &residual_out, &rms_weight, &act_scale, &B, &D, &scale_a}) check_same_device(input, *t, "every tensor");
    const float* scale_b_ptr = nullptr;
    int sb_stride = 0;
    if (scale_b.has_value()) {
        TORCH_CHECK(scale_b->scalar_type() == at::kFloat && scale_b->is_contiguous() && (scale_b->numel() == 1 || scale_b->numel() == n),
                    "scale_b must be float32 with 1 or n elements");
        check_same_device(input, *scale_b, "scale_b");
        scale_b_ptr = scale_b->data_ptr<float>();
        sb_stride = scale_b->numel() == 1 ? 0 : 1;
    }
    int d_dtype;
    const void* base_ptr = nullptr;
    const float* out_scale_ptr = nullptr;
    if (epilogue == HFRK_EPILOGUE_SWIGLU) {
        TORCH_CHECK(n % 2 == 0 && D.dim() == 2 && D.size(0) == m && D.size(1) == n / 2 && D.is_contiguous(), "D must be a contiguous [m, n/2] tensor");
        check_fp8(D, "D");
        TORCH_CHECK(out_scale.has_value() && out_scale->numel() == 1 && out_scale->scalar_type() == at::kFloat, "out_scale must be one float32");
        check_same_device(input, *out_scale, "out_scale");
        TORCH_CHECK(!base.has_value(), "base cannot be combined with the SwiGLU epilogue");
        TORCH_CHECK(intermediate_dtype == HFRK_F16 || intermediate_dtype == HFRK_BF16, "intermediate_dtype must be 0 (float16) or 1 (bfloat16)");
        d_dtype = (int)intermediate_dtype;
        out_scale_ptr = out_scale->data_ptr<float>();
    } else {
        TORCH_CHECK(D.dim() == 2 && D.size(0) == m && D.size(1) == n && D.is_contiguous(), "D must be a contiguous [m, n] tensor");
        d_dtype = dtype16(D, "D");
        if (base.has_value()) {
            TORCH_CHECK(base->sizes() == D.sizes() && base->is_contiguous() && base->scalar_type() == D.scalar_type(),
                        "base must be a contiguous tensor with D's shape and dtype");
            check_same_device(input, *base, "base");
            base_ptr = base->data_ptr();
        }
    }
    DeviceScope scope(input);
    return hfrk_skinny_gemm_rms_fused(input.data_ptr(), residual.data_ptr(), residual_out.data_ptr(), rms_weight.data_ptr(), (float)epsilon,
                                      act_scale.data_ptr<float>(), io, B.data_ptr(), D.data_ptr(), base_ptr, scale_a.data_ptr<float>(),
                                      scale_b_ptr, sb_stride, out_scale_ptr, (int)m, (int)n, (int)k, row_stride(B), d_dtype,
                                      (int)epilogue, nullptr, current_stream(input));
}

// The same on a weight in the load format of hfrk_pack_weight (no reference counterpart).
int64_t skinny_gemm_packed(at::Tensor& A, at::Tensor& B_packed, int64_t n, at::Tensor& D, const std::optional<at::Tensor>& base,
                           at::Tensor& scale_a, const std::optional<at::Tensor>& scale_b, const std::optional<at::Tensor>& out_scale,
                           int64_t epilogue, int64_t intermediate_dtype) {
    return gemm_fused_common(A, B_packed, true, n, D, base, scale_a, scale_b, out_scale, epilogue, intermediate_dtype);
}

// The linear layer's GEMM for any number of rows: D = base + scale_a x scale_b x A.B, base a [m, n] tensor or one [n] row.  Raises
// on a non-zero status.  No reference counterpart (its kernel stops at 32 rows, skinny_gemm_caller.cu:33-60).
void tiled_gemm(at::Tensor& A, at::Tensor& B, bool packed, int64_t n, at::Tensor& D, const std::optional<at::Tensor>& base,
                at::Tensor& scale_a, const std::optional<at::Tensor>& scale_b) {
    TORCH_CHECK(A.dim() == 2 && A.is_contiguous(), "A must be a contiguous [m, k] tensor");
    check_fp8(A, "A");
    check_fp8(B, "B");
    const int64_t m = A.size(0), k = A.size(1);
    TORCH_CHECK(n >= 1 && n < (int64_t(1) << 30) && m < (int64_t(1) << 30) && k < (int64_t(1) << 30), "m, n and k must fit 30 bits");
    if (packed) {
        const size_t plain = hfrk_packed_weight_bytes((int)n, (int)k), scaled = hfrk_packed_weight_bytes_scaled((int)n, (int)k);
        TORCH_CHECK(B.is_contiguous() && B.numel() > 0 && ((size_t)B.numel() == plain || (size_t)B.numel() == scaled),
                    "B must be the packed buffer of a [n, k] weight (pack_weight, pack_weight_scaled) with k = A.size(1)");
    } else {
        TORCH_CHECK(B.dim() == 2 && B.size(0) == k && B.size(1) == n && B.stride(0) == 1, "B must be [k, n] with unit stride along k");
    }
    TORCH_CHECK(D.dim() == 2 && D.size(0) == m && D.size(1) == n && D.is_contiguous(), "D must be a contiguous [m, n] tensor");
    const int d_dtype = dtype16(D, "D");
    TORCH_CHECK(scale_a.scalar_type() == at::kFloat && scale_a.is_contiguous() && (scale_a.numel() == 1 || scale_a.numel() == m),
                "scale_a must be float32 with 1 or m elements");
    check_same_device(A, B, "B");
    check_same_device(A, D, "D");
    check_same_device(A, scale_a, "scale_a");
    const float* scale_b_ptr = nullptr;
    int sb_stride = 0;
    if (scale_b.has_value()) {
        TORCH_CHECK(scale_b->scalar_type() == at::kFloat && scale_b->is_contiguous() && (scale_b->numel() == 1 || scale_b->numel() == n),
                    "scale_b must be float32 with 1 or n elements");
        check_same_device(A, *scale_b, "scale_b");
        scale_b_ptr = scale_b->data_ptr<float>();
        sb_stride = scale_b->numel() == 1 ? 0 : 1;
    }
    const void* base_ptr = nullptr;
    int base_stride = 0;
    if (base.has_value()) {
        const bool row = base->dim() == 1;
        TORCH_CHECK(base->is_contiguous() && base->scalar_type() == D.scalar_type() && (row ? base->size(0) == n : base->sizes() == D.sizes()),
                    "base must be a contiguous [n] or [m, n] tensor of D's dtype");
        check_same_device(A, *base, "base");
        base_ptr = base->data_ptr();
        base_stride = row ? 0 : (int)n;
    }
    if (m == 0) return;
    DeviceScope scope(A);
    const int sa_stride = scale_a.numel() == 1 ? 0 : 1, b_stride = packed ? (int)k : row_stride(B);
    const float* const sa = scale_a.data_ptr<float>();
    raise_on(hfrk_linear_gemm(A.data_ptr(), B.data_ptr(), packed ? 1 : 0, D.data_ptr(), base_ptr, base_stride, sa, sa_stride, scale_b_ptr,
                              sb_stride, (int)m, (int)n, (int)k, b_stride, d_dtype, current_stream(A)),
             "tiled_gemm");
}

// ---- whole calls as one operator ------------------------------------------------------------------------------------------
// What `Fp8Linear` and `skinny_gemm` do per call, allocations included.  A decode-sized call is a few microseconds of GPU work;
// as Python (argument checks, two allocations, two operators) its host side took longer than that: Fp8Linear of 16 rows
// 6144 x 4096 22.4 us per call against 11 us of kernels, skinny_gemm of 1 row 4096 x 4096 13.3 against 5.
// Both take only what is certain to run and return an undefined tensor (None in Python) or false for everything else; the Python
// wrapper then goes its general way, which converts, copies or raises.

bool one_float(const at::Tensor& t, const at::Tensor& like) {
    return t.numel() == 1 && t.scalar_type() == at::kFloat && t.device() == like.device();
}

bool float_vector(const at::Tensor& t, int64_t count, const at::Tensor& like) {
    return (t.numel() == 1 || t.numel() == count) && t.scalar_type() == at::kFloat && t.is_contiguous() && t.device() == like.device();
}

bool is_16bit(at::ScalarType t) { return t == at::kBFloat16 || t == at::kHalf; }

// input [..., k] 16-bit (quantised here: with input_scale, or per row when it is None) or fp8 with its scale(s); weight the
// row-major [n, k] fp8 tensor (n = -1) or the packed buffer of a weight of n rows; D = bias or residual + input . weight^T.
at::Tensor fp8_linear(const at::Tensor& input, const at::Tensor& weight, int64_t n, const std::optional<at::Tensor>& weight_scale,
                      const std::optional<at::Tensor>& input_scale, const std::optional<at::Tensor>& bias,
                      const std::optional<at::Tensor>& residual, std::optional<at::ScalarType> out_dtype) {
    const bool packed = n >= 0, quantised = input.scalar_type() == at::kFloat8_e4m3fn;
    if (!input.is_cuda() || input.dim() < 1 || input.numel() == 0 || !input.is_contiguous()) return {};
    if (!quantised && !is_16bit(input.scalar_type())) return {};
    if (weight.scalar_type() != at::kFloat8_e4m3fn || weight.device() != input.device()) return {};
    const int64_t k = input.size(-1), m = input.numel() / k;
    if (k >= (int64_t(1) << 24) || m >= (int64_t(1) << 24)) return {};
    const float* sb = nullptr;
    int sb_stride = 0, b_stride = (int)k;
    if (packed) {
        if (n < 1 || n >= (int64_t(1) << 24) || !weight.is_contiguous()) return {};
        const size_t plain = hfrk_packed_weight_bytes((int)n, (int)k), scaled = hfrk_packed_weight_bytes_scaled((int)n, (int)k);
        const size_t have = (size_t)weight.numel();
        if (plain == 0 || (have != plain && have != scaled)) return {};
        if (!weight_scale.has_value()) {  // the per-channel scales stored behind the packed bytes
            if (have == plain) return {};
            sb = reinterpret_cast<const float*>(static_cast<const uint8_t*>(weight.data_ptr()) + plain);
            sb_stride = 1;
        }
    } else {
        if (weight.dim() != 2 || weight.size(1) != k || weight.stride(1) != 1 || !weight_scale.has_value()) return {};
        n = weight.size(0);
        if (n < 1 || n >= (int64_t(1) << 24) || weight.stride(0) < k || weight.stride(0) >= (int64_t(1) << 30)) return {};
        b_stride = (int)weight.stride(0);
    }
    if (weight_scale.has_value()) {
        if (!float_vector(*weight_scale, n, input)) return {};
        sb = weight_scale->data_ptr<float>();
        sb_stride = weight_scale->numel() == 1 ? 0 : 1;
    }
    if (quantised && !input_scale.has_value()) return {};
    if (input_scale.has_value() && !(quantised ? float_vector(*input_scale, m, input) : one_float(*input_scale, input))) return {};
    if (!quantised && (k % 8 != 0 || k > 32768)) return {};
    const at::ScalarType dtype = out_dtype.value_or(quantised ? at::kBFloat16 : input.scalar_type());
    if (!is_16bit(dtype) || (bias.has_value() && residual.has_value())) return {};
    at::Tensor base;
    int base_stride = (int)n;
    if (residual.has_value()) {
        if (residual->numel() != m * n || !residual->is_contiguous() || residual->scalar_type() != dtype) return {};
        base = *residual;
    } else if (bias.has_value()) {
        if (bias->dim() != 1 || bias->size(0) != n || !bias->is_contiguous() || bias->scalar_type() != dtype) return {};
        base = *bias;
        base_stride = 0;
    }
    if (base.defined() && base.device() != input.device()) return {};

    DeviceScope scope(input);
    void* const stream = current_stream(input);
    at::DimVector sizes(input.sizes());
    sizes.back() = n;
    at::Tensor out = at::empty(sizes, input.options().dtype(dtype));
    const void* a = input.data_ptr();
    const float* sa = nullptr;
    int sa_stride = 0;
    at::Tensor scratch;  // the quantised rows, then their scales
    if (input_scale.has_value()) {
        sa = input_scale->data_ptr<float>();
        sa_stride = input_scale->numel() == 1 ? 0 : 1;
    }
    if (!quantised) {
        const int64_t bytes = (m * k + 15) / 16 * 16;
        scratch = at::empty({bytes + (sa ? 0 : 4 * m)}, input.options().dtype(at::kByte));
        uint8_t* const q = static_cast<uint8_t*>(scratch.data_ptr());
        float* const row_scales = reinterpret_cast<float*>(q + bytes);
        if (hfrk_quantize_fp8(a, sa, q, sa ? nullptr : row_scales, (int)m, (int)k, input.scalar_type() == at::kBFloat16 ? HFRK_BF16 : HFRK_F16,
                              stream) != HFRK_SUCCESS)
            return {};
        a = q;
        if (!sa) {
            sa = row_scales;
            sa_stride = 1;
        }
    }
    const void* const base_ptr = base.defined() ? base.data_ptr() : nullptr;
    const int d_dtype = dtype == at::kBFloat16 ? HFRK_BF16 : HFRK_F16;
    const int status = hfrk_linear_gemm(a, weight.data_ptr(), packed ? 1 : 0, out.data_ptr(), base_ptr, base_stride, sa, sa_stride, sb,
                                        sb_stride, (int)m, (int)n, (int)k, b_stride, d_dtype, stream);
    return status == HFRK_SUCCESS ? out : at::Tensor();
}

// The operands `skinny_gemm` takes with nothing to convert or report: a row-major weight whose rows are whole 256-byte chunks.
bool plain_gemm_operands(const at::Tensor& A, const at::Tensor& B, const at::Tensor& scale) {
    return A.is_cuda() && A.dim() == 2 && B.dim() == 2 && A.scalar_type() == at::kFloat8_e4m3fn && B.scalar_type() == at::kFloat8_e4m3fn &&
           A.is_contiguous() && B.size(0) == A.size(1) && B.stride(0) == 1 && A.size(0) >= 1 && A.size(0) <= HFRK_GEMM_MAX_M &&
           A.size(1) >= 256 && A.size(1) % 256 == 0 && A.size(1) < (int64_t(1) << 24) && B.size(1) >= 2 && B.size(1) % 2 == 0 &&
           B.size(1) < (int64_t(1) << 24) && B.stride(1) >= A.size(1) && B.stride(1) < (int64_t(1) << 30) && B.device() == A.device() &&
           one_float(scale, A);
}

int plain_gemm(const at::Tensor& A, const at::Tensor& B, const at::Tensor& scale, const at::Tensor& D, bool accumulate) {
    return hfrk_skinny_gemm_ex(A.data_ptr(), B.data_ptr(), D.data_ptr(), scale.data_ptr<float>(), 0, nullptr, 0, (int)A.size(0),
                               (int)B.size(1), (int)A.size(1), (int)B.stride(1), dtype16(D, "D"), accumulate ? 1 : 0, nullptr,
                               current_stream(A));
}

// A new float16 tensor: written whole, where the reference's wrapper clears one and accumulates into it (wrapped.py:119).
at::Tensor skinny_gemm_new(const at::Tensor& A, const at::Tensor& B, const at::Tensor& scale) {
    if (!plain_gemm_operands(A, B, scale)) return {};
    DeviceScope scope(A);
    at::Tensor D = at::empty({A.size(0), B.size(1)}, A.options().dtype(at::kHalf));
    return plain_gemm(A, B, scale, D, false) == HFRK_SUCCESS ? D : at::Tensor();
}

bool skinny_gemm_into(const at::Tensor& A, const at::Tensor& B, const at::Tensor& scale, at::Tensor& D) {
    if (!plain_gemm_operands(A, B, scale) || D.dim() != 2 || D.size(0) != A.size(0) || D.size(1) != B.size(1) || !D.is_contiguous() ||
        !is_16bit(D.scalar_type()) || D.device() != A.device())
        return false;
    DeviceScope scope(A);
    return plain_gemm(A, B, scale, D, true) == HFRK_SUCCESS;
}

// The fused decoder MLP block (combined_ops/llama_mlp.py) as one operator: its Python side took about 35 us per call, the block of 8 rows
// of 4096 x 14336 35 us of kernels and that of one row of 2048 x 6144 less than half of it.  residual_out <- input + residual (it may be
// `residual`), input_copy <- input, and the block's output, into `output` where one is given.  Weights are [k, n] views or (n >= 0) packed buffers.
// False, with nothing launched, for everything that the wrappers would convert, copy or refuse.  memory: scratch, and behind it the workspace of
// hfrk_llama_mlp_owned; without it scratch is allocated and the workspace is the stream's.
bool llama_mlp(const at::Tensor& input, const at::Tensor& residual, at::Tensor& residual_out, const std::optional<at::Tensor>& input_copy,
               const at::Tensor& rms_weight, double epsilon, const at::Tensor& gate_up, int64_t gate_up_n, const at::Tensor& gate_up_input_scale,
               const at::Tensor& gate_up_output_scale, const at::Tensor& down, int64_t down_n, const at::Tensor& down_input_scale,
               const at::Tensor& down_output_scale, bool add_residual, at::Tensor& output, const std::optional<at::Tensor>& memory) {
    if (!input.is_cuda() || input.dim() != 2 || !is_16bit(input.scalar_type())) return false;
    const int64_t m = input.size(0), hidden = input.size(1);
    auto like_input = [&](const at::Tensor& t) {
        return t.is_contiguous() && t.sizes() == input.sizes() && t.scalar_type() == input.scalar_type() && t.device() == input.device();
    };
    if (m < 1 || m > HFRK_GEMM_MAX_M || hidden < 256 || hidden % 256 != 0 || hidden > 32768) return false;
    if (!like_input(input) || !like_input(residual) || !like_input(residual_out) || !like_input(output)) return false;
    if (input_copy.has_value() && !like_input(*input_copy)) return false;
    // copied in first and added to afterwards, as the general way has it, the residual would be the input (overlaps are the C entry's to refuse)
    if (input_copy.has_value() && residual.data_ptr() == input_copy->data_ptr() && input.data_ptr() != residual.data_ptr()) return false;
    if (at::GradMode::is_enabled() && (input.requires_grad() || residual.requires_grad())) return false;
    if (rms_weight.dim() != 1 || rms_weight.size(0) != hidden || !rms_weight.is_contiguous() || rms_weight.scalar_type() != input.scalar_type() ||
        rms_weight.device() != input.device() || !(epsilon > 0))
        return false;
    for (const at::Tensor* t : {&gate_up_input_scale, &gate_up_output_scale, &down_input_scale, &down_output_scale})
        if (!one_float(*t, input)) return false;
    // a weight's columns, or -1 where it is none of `k` rows that the GEMMs read as it is
    auto columns = [&](const at::Tensor& w, int64_t n, int64_t k) -> int64_t {
        if (w.scalar_type() != at::kFloat8_e4m3fn || w.device() != input.device()) return -1;
        if (n >= 0) {
            if (n < 1 || n >= (int64_t(1) << 24) || !w.is_contiguous()) return -1;
            const size_t plain = hfrk_packed_weight_bytes((int)n, (int)k), have = (size_t)w.numel();
            return plain != 0 && (have == plain || have == hfrk_packed_weight_bytes_scaled((int)n, (int)k)) ? n : -1;
        }
        if (w.dim() != 2 || w.size(0) != k || w.stride(0) != 1 || w.size(1) < 2 || w.size(1) >= (int64_t(1) << 24) || w.stride(1) < k ||
            w.stride(1) >= (int64_t(1) << 30))
            return -1;
        return w.size(1);
    };
    const int64_t n = columns(gate_up, gate_up_n, hidden), inter = n / 2;
    if (n < 512 || inter % 256 != 0 || n % 2 != 0 || columns(down, down_n, inter) != hidden) return false;

    DeviceScope scope(input);
    const size_t scratch_bytes = hfrk_llama_mlp_scratch_bytes((int)m, (int)hidden, (int)inter);
    if (memory.has_value() && (memory->scalar_type() != at::kByte || !memory->is_contiguous() || memory->device() != input.device() ||
                               (size_t)memory->numel() < scratch_bytes))
        return false;
    at::Tensor scratch = memory.has_value() ? *memory : at::empty({(int64_t)scratch_bytes}, input.options().dtype(at::kByte));
    uint8_t* const workspace = memory.has_value() ? scratch.data_ptr<uint8_t>() + scratch_bytes : nullptr;
    int launched = 0;
    const int status = hfrk_llama_mlp_owned(
        input.data_ptr(), residual.data_ptr(), residual_out.data_ptr(), input_copy.has_value() ? input_copy->data_ptr() : nullptr,
        rms_weight.data_ptr(), (float)epsilon, gate_up_input_scale.data_ptr<float>(), gate_up.data_ptr(), gate_up_n >= 0 ? 1 : 0,
        gate_up_n >= 0 ? (int)hidden : (int)gate_up.stride(1), gate_up_output_scale.data_ptr<float>(), down_input_scale.data_ptr<float>(),
        down.data_ptr(), down_n >= 0 ? 1 : 0, down_n >= 0 ? (int)inter : (int)down.stride(1), down_output_scale.data_ptr<float>(),
        add_residual ? 1 : 0, output.data_ptr(), scratch.data_ptr(), workspace, workspace ? (size_t)scratch.numel() - scratch_bytes : 0, (int)m,
        (int)hidden, (int)inter, input.scalar_type() == at::kBFloat16 ? HFRK_BF16 : HFRK_F16, &launched, current_stream(input));
    if (launched) raise_on(status, "llama_mlp");
    return status == HFRK_SUCCESS;
}

// The row kernels beside the GEMMs as their wrappers are usually called: no buffer to clear and the launcher's own choice of threads.  In Python the
// checks, two to four allocations and the operator took 8 to 10 us a call, the kernels 2 to 4; now 5.5 to 6.3.  A tensor that requires a gradient changes
// nothing: the general operators return no tensor and record nothing either.
bool plain_rows(const at::Tensor& x) {
    return x.is_cuda() && x.dim() == 2 && is_16bit(x.scalar_type()) && x.is_contiguous() && x.size(1) > 0 && x.size(0) < (int64_t(1) << 24) &&
           x.size(1) < (int64_t(1) << 24);
}

bool plain_rms(const at::Tensor& input, const at::Tensor& residual, const at::Tensor& weight, double epsilon) {
    return plain_rows(input) && plain_rows(residual) && residual.sizes() == input.sizes() && residual.scalar_type() == input.scalar_type() &&
           residual.device() == input.device() && weight.dim() == 1 && weight.size(0) == input.size(1) && weight.is_contiguous() &&
           weight.scalar_type() == input.scalar_type() && weight.device() == input.device() && epsilon > 0;
}

// Rows that the dynamic kernels take: whole 16-byte pieces, held in registers.
bool dynamic_columns(int64_t cols) { return cols % 8 == 0 && cols <= 32768; }

at::Tensor residual_rms_new(const at::Tensor& input, at::Tensor& residual, const at::Tensor& weight, double epsilon, const std::optional<at::Tensor>& scale) {
    if (!plain_rms(input, residual, weight, epsilon) || (scale.has_value() && !one_float(*scale, input))) return {};
    DeviceScope scope(input);
    const int io = dtype16(input, "input");
    at::Tensor output = at::empty(input.sizes(), input.options().dtype(scale.has_value() ? at::kFloat8_e4m3fn : input.scalar_type()));
    return hfrk_residual_rms(input.data_ptr(), residual.data_ptr(), weight.data_ptr(), scale.has_value() ? scale->data_ptr<float>() : nullptr, (float)epsilon,
                             output.data_ptr(), nullptr, (int)input.size(0), (int)input.size(1), 0, io, scale.has_value() ? HFRK_FP8_E4M3FN : io, 0, 0,
                             current_stream(input)) == HFRK_SUCCESS
               ? output
               : at::Tensor();
}

std::tuple<at::Tensor, at::Tensor> residual_rms_dynamic_new(const at::Tensor& input, at::Tensor& residual, const at::Tensor& weight, double epsilon) {
    if (!plain_rms(input, residual, weight, epsilon) || !dynamic_columns(input.size(1))) return {};
    DeviceScope scope(input);
    at::Tensor output = at::empty(input.sizes(), input.options().dtype(at::kFloat8_e4m3fn));
    at::Tensor scales = at::empty({input.size(0)}, input.options().dtype(at::kFloat));
    if (hfrk_residual_rms_dynamic(input.data_ptr(), residual.data_ptr(), weight.data_ptr(), (float)epsilon, output.data_ptr(), scales.data_ptr<float>(), nullptr,
                                  (int)input.size(0), (int)input.size(1), 0, dtype16(input, "input"), current_stream(input)) != HFRK_SUCCESS)
        return {};
    return {output, scales};
}

at::Tensor swiglu_new(const at::Tensor& gate_up, const at::Tensor& scale) {
    if (!plain_rows(gate_up) || gate_up.size(1) % 2 != 0 || !one_float(scale, gate_up)) return {};
    DeviceScope scope(gate_up);
    const int64_t rows = gate_up.size(0), cols = gate_up.size(1) / 2;
    at::Tensor output = at::empty({rows, cols}, gate_up.options().dtype(at::kFloat8_e4m3fn));
    return hfrk_swiglu(gate_up.data_ptr(), scale.data_ptr<float>(), output.data_ptr(), nullptr, (int)rows, (int)cols, 0, dtype16(gate_up, "gate_up"), 0, 0,
                       current_stream(gate_up)) == HFRK_SUCCESS
               ? output
               : at::Tensor();
}

std::tuple<at::Tensor, at::Tensor> swiglu_dynamic_new(const at::Tensor& gate_up) {
    if (!plain_rows(gate_up) || gate_up.size(1) % 2 != 0 || !dynamic_columns(gate_up.size(1) / 2)) return {};
    DeviceScope scope(gate_up);
    const int64_t rows = gate_up.size(0), cols = gate_up.size(1) / 2;
    at::Tensor output = at::empty({rows, cols}, gate_up.options().dtype(at::kFloat8_e4m3fn));
    at::Tensor scales = at::empty({rows}, gate_up.options().dtype(at::kFloat));
    if (hfrk_swiglu_dynamic(gate_up.data_ptr(), output.data_ptr(), scales.data_ptr<float>(), nullptr, (int)rows, (int)cols, 0, dtype16(gate_up, "gate_up"),
                            current_stream(gate_up)) != HFRK_SUCCESS)
        return {};
    return {output, scales};
}

bool is_byte_tensor(const at::Tensor& t) {
    return t.scalar_type() == at::kByte || t.scalar_type() == at::kFloat8_e4m3fn || t.scalar_type() == at::kFloat8_e4m3fnuz;
}

// The fused GEMM for tracers: same call as skinny_gemm_fused / skinny_gemm_packed, but a status other than 0 raises
// instead of being returned.  An operator that returns an integer cannot be part of a traced graph; one that returns
// nothing can.
void skinny_gemm_checked(at::Tensor& A, at::Tensor& B, bool packed, int64_t n, at::Tensor& D, const std::optional<at::Tensor>& base,
                         at::Tensor& scale_a, const std::optional<at::Tensor>& scale_b, const std::optional<at::Tensor>& out_scale,
                         int64_t epilogue, int64_t intermediate_dtype) {
    TORCH_CHECK(packed || B.dim() == 2, "B must be [k, n] with unit stride along k");
    raise_on((int)gemm_fused_common(A, B, packed, packed ? n : B.size(1), D, base, scale_a, scale_b, out_scale, epilogue, intermediate_dtype),
             "skinny_gemm_checked");
}

// Row-major [n, k] fp8 weight -> packed load format; src_format 1 re-encodes e4m3fnuz values as e4m3fn on the way.
void pack_weight(at::Tensor& src, at::Tensor& dst, int64_t src_format) {
    TORCH_CHECK(src.dim() == 2 && src.stride(1) == 1 && is_byte_tensor(src), "src must be a [n, k] one-byte tensor with unit stride along k");
    TORCH_CHECK(src.size(0) < (int64_t(1) << 30) && src.size(1) < (int64_t(1) << 30), "n and k must fit 30 bits");
    const int n = (int)src.size(0), k = (int)src.size(1);
    TORCH_CHECK(is_byte_tensor(dst) && dst.is_contiguous() && (size_t)dst.numel() == hfrk_packed_weight_bytes(n, k) && dst.numel() > 0,
                "dst must be a contiguous one-byte tensor of hfrk_packed_weight_bytes(n, k) elements (k % 256 == 0)");
    check_same_device(src, dst, "dst");
    DeviceScope scope(src);
    raise_on(hfrk_pack_weight(src.data_ptr(), (int)src.stride(0), (int)src_format, dst.data_ptr(), n, k, current_stream(src)), "pack_weight");
}

// The same with the weight's per-output-channel scales stored behind the packed bytes (one allocation per layer).
void pack_weight_scaled(at::Tensor& src, at::Tensor& scales, at::Tensor& dst, int64_t src_format) {
    TORCH_CHECK(src.dim() == 2 && src.stride(1) == 1 && is_byte_tensor(src), "src must be a [n, k] one-byte tensor with unit stride along k");
    TORCH_CHECK(src.size(0) < (int64_t(1) << 30) && src.size(1) < (int64_t(1) << 30), "n and k must fit 30 bits");
    const int n = (int)src.size(0), k = (int)src.size(1);
    TORCH_CHECK(scales.scalar_type() == at::kFloat && scales.is_contiguous() && scales.numel() == n, "scales must be n contiguous float32 values");
    TORCH_CHECK(is_byte_tensor(dst) && dst.is_contiguous() && (size_t)dst.numel() == hfrk_packed_weight_bytes_scaled(n, k) && dst.numel() > 0,
                "dst must be a contiguous one-byte tensor of hfrk_packed_weight_bytes_scaled(n, k) elements (k % 256 == 0)");
    check_same_device(src, dst, "dst");
    check_same_device(src, scales, "scales");
    DeviceScope scope(src);
    raise_on(hfrk_pack_weight_scaled(src.data_ptr(), (int)src.stride(0), (int)src_format, scales.data_ptr<float>(), dst.data_ptr(), n, k,
                                     current_stream(src)), "pack_weight_scaled");
}

void unpack_weight(at::Tensor& src, at::Tensor& dst) {
    TORCH_CHECK(dst.dim() == 2 && dst.stride(1) == 1 && is_byte_tensor(dst), "dst must be a [n, k] one-byte tensor with unit stride along k");
    TORCH_CHECK(dst.size(0) < (int64_t(1) << 30) && dst.size(1) < (int64_t(1) << 30), "n and k must fit 30 bits");
    const int n = (int)dst.size(0), k = (int)dst.size(1);
    TORCH_CHECK(is_byte_tensor(src) && src.is_contiguous() && src.numel() > 0 &&
                    ((size_t)src.numel() == hfrk_packed_weight_bytes(n, k) || (size_t)src.numel() == hfrk_packed_weight_bytes_scaled(n, k)),
                "src must be a contiguous one-byte tensor of hfrk_packed_weight_bytes(n, k) elements (k % 256 == 0), or that plus its scales");
    check_same_device(src, dst, "dst");
    DeviceScope scope(src);
    raise_on(hfrk_unpack_weight(src.data_ptr(), dst.data_ptr(), (int)dst.stride(0), n, k, current_stream(src)), "unpack_weight");
}

// e4m3fnuz bytes -> e4m3fn bytes with the same values (dst may be src).
void reencode_fnuz(at::Tensor& src, at::Tensor& dst) {
    TORCH_CHECK(is_byte_tensor(src) && is_byte_tensor(dst) && src.is_contiguous() && dst.is_contiguous() && src.numel() == dst.numel(),
                "src and dst must be contiguous one-byte tensors of the same size");
    check_same_device(src, dst, "dst");
    DeviceScope scope(src);
    raise_on(hfrk_reencode_fnuz(src.data_ptr(), dst.data_ptr(), (size_t)src.numel(), current_stream(src)), "reencode_fnuz");
}

}  // namespace

TORCH_LIBRARY(_HFRK_C, ops) {
    ops.def("increment(Tensor! x) -> ()");
    ops.impl("increment", c10::kCUDA, &increment);

    ops.def(
        "residual_rms(Tensor input, Tensor! residual, Tensor weight, Tensor scale_tensor, float epsilon, Tensor! "
        "output, Tensor! next_buffer, int num_threads, bool force_scalar) -> ()");
    ops.impl("residual_rms", c10::kCUDA, &residual_rms);

    ops.def(
        "swiglu(Tensor gate_up, Tensor scale_tensor, Tensor! output, Tensor! next_buffer, int num_threads, "
        "bool force_scalar) -> ()");
    ops.impl("swiglu", c10::kCUDA, &swiglu);

    ops.def(
        "skinny_gemm_tb(Tensor A, Tensor B, Tensor! D, Tensor scale_tensor, int split_k, int A_producers, "
        "int B_producers, int consumers, int a_lanes, int b_lanes, int qsize, int op_m, int ops) -> int");
    ops.impl("skinny_gemm_tb", c10::kCUDA, &skinny_gemm_tb);

    ops.def("skinny_gemm_scaled(Tensor A, Tensor B, Tensor! D, Tensor scale_a, Tensor scale_b, bool accumulate) -> int");
    ops.impl("skinny_gemm_scaled", c10::kCUDA, &skinny_gemm_scaled);

    ops.def(
        "skinny_gemm_fused(Tensor A, Tensor B, Tensor! D, Tensor? base, Tensor scale_a, Tensor? scale_b, "
        "Tensor? out_scale, int epilogue, int intermediate_dtype) -> int");
    ops.impl("skinny_gemm_fused", c10::kCUDA, &skinny_gemm_fused);
    ops.def(
        "skinny_gemm_rms_fused(Tensor input, Tensor residual, Tensor! residual_out, Tensor rms_weight, float epsilon, "
        "Tensor act_scale, Tensor B, Tensor! D, Tensor? base, Tensor scale_a, Tensor? scale_b, Tensor? out_scale, "
        "int epilogue, int intermediate_dtype) -> int");
    ops.impl("skinny_gemm_rms_fused", c10::kCUDA, &skinny_gemm_rms_fused);

    ops.def(
        "skinny_gemm_packed(Tensor A, Tensor B_packed, int n, Tensor! D, Tensor? base, Tensor scale_a, Tensor? scale_b, "
        "Tensor? out_scale, int epilogue, int intermediate_dtype) -> int");
    ops.impl("skinny_gemm_packed", c10::kCUDA, &skinny_gemm_packed);

    ops.def(
        "skinny_gemm_checked(Tensor A, Tensor B, bool packed, int n, Tensor! D, Tensor? base, Tensor scale_a, Tensor? scale_b, "
        "Tensor? out_scale, int epilogue, int intermediate_dtype) -> ()");
    ops.impl("skinny_gemm_checked", c10::kCUDA, &skinny_gemm_checked);

    ops.def(
        "tiled_gemm(Tensor A, Tensor B, bool packed, int n, Tensor! D, Tensor? base, Tensor scale_a, Tensor? scale_b) -> ()");
    ops.impl("tiled_gemm", c10::kCUDA, &tiled_gemm);

    ops.def("pack_weight(Tensor src, Tensor! dst, int src_format) -> ()");
    ops.impl("pack_weight", c10::kCUDA, &pack_weight);
    ops.def("pack_weight_scaled(Tensor src, Tensor scales, Tensor! dst, int src_format) -> ()");
    ops.impl("pack_weight_scaled", c10::kCUDA, &pack_weight_scaled);
    ops.def("unpack_weight(Tensor src, Tensor! dst) -> ()");
    ops.impl("unpack_weight", c10::kCUDA, &unpack_weight);
    ops.def("reencode_fnuz(Tensor src, Tensor! dst) -> ()");
    ops.impl("reencode_fnuz", c10::kCUDA, &reencode_fnuz);

    ops.def(
        "residual_rms_dynamic(Tensor input, Tensor! residual, Tensor weight, float epsilon, Tensor! output, "
        "Tensor! scales, Tensor! next_buffer) -> ()");
    ops.impl("residual_rms_dynamic", c10::kCUDA, &residual_rms_dynamic);

    ops.def("swiglu_dynamic(Tensor gate_up, Tensor! output, Tensor! scales, Tensor! next_buffer) -> ()");
    ops.impl("swiglu_dynamic", c10::kCUDA, &swiglu_dynamic);

    // Outputs carry no autograd history, as those of the operators that write into a tensor of the caller's.
    ops.def(
        "fp8_linear(Tensor input, Tensor weight, int n, Tensor? weight_scale, Tensor? input_scale, Tensor? bias, Tensor? residual, "
        "ScalarType? out_dtype) -> Tensor");
    ops.impl("fp8_linear", c10::kCUDA, &fp8_linear);
    ops.impl("fp8_linear", torch::dispatch(c10::DispatchKey::Autograd, torch::CppFunction::makeFallthrough()));
    ops.def("skinny_gemm_new(Tensor A, Tensor B, Tensor scale) -> Tensor");
    ops.impl("skinny_gemm_new", c10::kCUDA, &skinny_gemm_new);
    ops.impl("skinny_gemm_new", torch::dispatch(c10::DispatchKey::Autograd, torch::CppFunction::makeFallthrough()));
    ops.def("skinny_gemm_into(Tensor A, Tensor B, Tensor scale, Tensor! D) -> bool");
    ops.impl("skinny_gemm_into", c10::kCUDA, &skinny_gemm_into);

    ops.def(
        "llama_mlp(Tensor input, Tensor residual, Tensor(a!) residual_out, Tensor(b!)? input_copy, Tensor rms_weight, float epsilon, Tensor gate_up, "
        "int gate_up_n, Tensor gate_up_input_scale, Tensor gate_up_output_scale, Tensor down, int down_n, Tensor down_input_scale, "
        "Tensor down_output_scale, bool add_residual, Tensor(c!) output, Tensor(d!)? memory=None) -> bool");
    ops.impl("llama_mlp", c10::kCUDA, &llama_mlp);
    ops.impl("llama_mlp", torch::dispatch(c10::DispatchKey::Autograd, torch::CppFunction::makeFallthrough()));

    ops.def("residual_rms_new(Tensor input, Tensor(a!) residual, Tensor weight, float epsilon, Tensor? scale) -> Tensor");
    ops.impl("residual_rms_new", c10::kCUDA, &residual_rms_new);
    ops.def("residual_rms_dynamic_new(Tensor input, Tensor(a!) residual, Tensor weight, float epsilon) -> (Tensor, Tensor)");
    ops.impl("residual_rms_dynamic_new", c10::kCUDA, &residual_rms_dynamic_new);
    ops.def("swiglu_new(Tensor gate_up, Tensor scale) -> Tensor");
    ops.impl("swiglu_new", c10::kCUDA, &swiglu_new);
    ops.def("swiglu_dynamic_new(Tensor gate_up) -> (Tensor, Tensor)");
    ops.impl("swiglu_dynamic_new", c10::kCUDA, &swiglu_dynamic_new);
    for (const char* name : {"residual_rms_new", "residual_rms_dynamic_new", "swiglu_new", "swiglu_dynamic_new"})
        ops.impl(name, torch::dispatch(c10::DispatchKey::Autograd, torch::CppFunction::makeFallthrough()));

    ops.def("quantize_fp8(Tensor input, Tensor? scale_tensor, Tensor! output, Tensor! scales) -> ()");
    ops.impl("quantize_fp8", c10::kCUDA, &quantize_fp8);
}

// nothing_intercepts() -> bool: whether an operator called now, on plain tensors, runs its kernel and is seen by nobody else.  Whatever
// records, batches or replaces calls (torch.jit.trace, functorch's transforms, dispatch modes and fake tensors, pre-dispatch tracing,
// functionalisation) does so by a dispatch key that it includes for the thread.
static PyObject* nothing_intercepts(PyObject*, PyObject*) {
    const bool none = (c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set).empty();
    return PyBool_FromLong(none);
}

// `import hf_rocm_kernels._HFRK_C` loads this library and thereby runs the registration above.
PyMODINIT_FUNC PyInit__HFRK_C(void) {
    static PyMethodDef methods[] = {{"nothing_intercepts", nothing_intercepts, METH_NOARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
    static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_HFRK_C", nullptr, 0, methods};
    return PyModule_Create(&module);
}
