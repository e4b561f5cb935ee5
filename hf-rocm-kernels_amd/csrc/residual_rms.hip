// residual <- input + residual;  output <- rmsnorm(residual) * weight [ / scale -> fp8 e4m3fn ];  next_buffer <- 0
//
// Replaces csrc/op_src/residual_rms/residual_rms_dispatch.cu:8-63 and its two kernels
// (residual_rms_scalar.cu:11-74, residual_rms_vectorized.cu:13-172).  One workgroup per row.  The summed row is
// kept in registers between the two passes (the reference parks it in a 32 KB LDS array), the sum of squares is
// reduced in registers inside each wavefront and by one LDS exchange of <= 16 floats between wavefronts,
// and every thread adds those partials in the same order, so the normaliser is identical for the whole row.
//
// Arithmetic (same points of rounding as the reference's torch functions, operators/residual_rms/reference.py:7-36):
//   z   = round16(float(input) + float(residual))            -> stored to residual, bit-exact with a torch add
//   r   = rsqrt(mean(float(z)^2) + eps)                      fp32
//   16-bit output:  round16( float(round16(float(z) * r)) * float(weight) )
//   fp8 output:     e4m3fn( clamp( float(z) * r * float(weight) * (1/scale), +-448 ) )   no 16-bit detour, as in
//                   the reference's vectorised kernel (residual_rms_vectorized.cu:124-135)
#include "hfrk_internal.h"

namespace hfrk {

constexpr int kRmsMaxThreads = 1024;

// From this many values on the input is read past the caches, which leaves their room (256 MB behind the L2s) to the residual, the weight
// and the output.  Measured with both reads on fp16, us, kept / past.  Calls on buffers that change: 2048 x 4096 10.2 / 11.2,
// 2048 x 8192 18.3 / 19.7, 1536 x 16384 30.4 / 28.6, 1792 x 16384 36.9 / 33.4, 2048 x 16384 43.2 / 37.9, 4096 x 16384 83.2 / 80.3.  With a
// kernel in front that has just written the input, both: 2048 x 8192 30.9 / 31.5, 1536 x 16384 44.6 / 44.8, 4096 x 8192 66.2 / 59.0,
// 4096 x 16384 128.5 / 125.0.  One set of buffers again and again, nothing else between: 1965 x 11328 25.1 / 27.7, 2048 x 16384 35.5 / 38.5,
// 4096 x 16384 72.1 / 72.4.  At decode sizes reading past them cost an eager MLP block of 1 to 16 rows of 4096 0.4 us of 32.
constexpr long kReadOnceFrom = 28L << 20;

__device__ __forceinline__ void zero_next_buffer_row(uint16_t* next_buffer, int buffer_cols) {
    if (buffer_cols <= 0) return;
    uint16_t* const row = next_buffer + (long)blockIdx.x * buffer_cols;
    // 16-byte stores where the row allows it, element stores for the ragged ends
    const uintptr_t addr = reinterpret_cast<uintptr_t>(row);
    int head = (int)(((16 - (addr & 15)) & 15) >> 1);
    if (head > buffer_cols) head = buffer_cols;
    const int body = (buffer_cols - head) >> 3;
    for (int i = threadIdx.x; i < head; i += blockDim.x) row[i] = 0;
    uint4* const vec = reinterpret_cast<uint4*>(row + head);
    for (int i = threadIdx.x; i < body; i += blockDim.x) vec[i] = make_uint4(0, 0, 0, 0);
    for (int i = head + body * 8 + threadIdx.x; i < buffer_cols; i += blockDim.x) row[i] = 0;
}

// 8 elements (16 bytes) per thread per iteration, ITERS iterations cached in registers: cols <= 8*blockDim*ITERS.
// READ_ONCE: the input is read past the caches (kReadOnceFrom).
// INTO: the residual is read from residual_in, which stays as it is unless it is `residual` itself, and input_copy, where not null,
// becomes a copy of the input.  Every thread has read its pieces of the inputs before it writes any, and nobody else's: either may be its
// own source.  Two kernels call this: with the further pointers and without __restrict__ the four-piece instances of the plain one take 62
// to 69 registers instead of 60 to 64, and beyond 64 a compute unit holds one workgroup of 16 waves instead of two.
template <int DT, bool FP8_OUT, int ITERS, bool READ_ONCE, bool INTO>
__device__ __forceinline__ void residual_rms_vec(
    const uint16_t* input, const uint16_t* residual_in, uint16_t* residual, uint16_t* input_copy, const uint16_t* weight,
    const float* scale_tensor, void* output, uint16_t* next_buffer, float epsilon, int cols, int buffer_cols) {
    __shared__ __align__(16) float red[16];
    const long row_off = (long)blockIdx.x * cols;
    const uint32_t row_bytes = (uint32_t)cols * 2u;
    const __amdgpu_buffer_rsrc_t rin = make_rsrc(input + row_off, row_bytes), rres = make_rsrc(residual + row_off, row_bytes),
                                 rweight = make_rsrc(weight, row_bytes);
    const __amdgpu_buffer_rsrc_t rres_in = INTO ? make_rsrc(residual_in + row_off, row_bytes) : rres;
    const __amdgpu_buffer_rsrc_t rout = FP8_OUT ? make_rsrc(static_cast<uint8_t*>(output) + row_off, (uint32_t)cols)
                                                : make_rsrc(static_cast<uint16_t*>(output) + row_off, row_bytes);
    uint4 a[ITERS], z[ITERS], wreg[ITERS];
    float ssq = 0.f;
    // Everything both passes need is requested now, so that the kernel pays one memory latency.
    float scale = 1.f;
    if constexpr (FP8_OUT) scale = scale_tensor[0];
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
        const int v = threadIdx.x + it * blockDim.x;
        a[it] = load_piece<READ_ONCE>(rin, v);
        z[it] = load_piece(rres_in, v);
    }
#pragma unroll
    for (int it = 0; it < ITERS; ++it) wreg[it] = load_piece(rweight, threadIdx.x + it * blockDim.x);
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
        z[it] = rms_add_square<DT>(a[it], z[it], ssq);
        store_piece(rres, threadIdx.x + it * blockDim.x, z[it]);
    }
    if (INTO && input_copy) {
        const __amdgpu_buffer_rsrc_t rcopy = make_rsrc(input_copy + row_off, row_bytes);
#pragma unroll
        for (int it = 0; it < ITERS; ++it) store_piece(rcopy, threadIdx.x + it * blockDim.x, a[it]);
    }
    const float total = block_sum(ssq, red);
    const float norm = rsqrtf(total / (float)cols + epsilon);
    const float inv_scale = 1.f / scale;

#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
        const int v = threadIdx.x + it * blockDim.x;
        const uint4 w = wreg[it];
        const uint32_t zw[4] = {z[it].x, z[it].y, z[it].z, z[it].w}, ww[4] = {w.x, w.y, w.z, w.w};
        if constexpr (FP8_OUT) {
            store_fp8_piece(rout, v, rms_scale_to_fp8<DT>(z[it], w, norm, inv_scale));
        } else {
            uint32_t ow[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint16_t nl = store16<DT>(load16<DT>((uint16_t)(zw[j] & 0xffff)) * norm);
                const uint16_t nh = store16<DT>(load16<DT>((uint16_t)(zw[j] >> 16)) * norm);
                const uint16_t ol = store16<DT>(load16<DT>(nl) * load16<DT>((uint16_t)(ww[j] & 0xffff)));
                const uint16_t oh = store16<DT>(load16<DT>(nh) * load16<DT>((uint16_t)(ww[j] >> 16)));
                ow[j] = (uint32_t)ol | ((uint32_t)oh << 16);
            }
            store_piece(rout, v, make_uint4(ow[0], ow[1], ow[2], ow[3]));
        }
    }
    zero_next_buffer_row(next_buffer, buffer_cols);
}

template <int DT, bool FP8_OUT, int ITERS, bool READ_ONCE>
__global__ void __launch_bounds__(kRmsMaxThreads) residual_rms_vec_kernel(
    const uint16_t* __restrict__ input, uint16_t* __restrict__ residual, const uint16_t* __restrict__ weight,
    const float* __restrict__ scale_tensor, void* __restrict__ output, uint16_t* __restrict__ next_buffer,
    float epsilon, int cols, int buffer_cols) {
    residual_rms_vec<DT, FP8_OUT, ITERS, READ_ONCE, false>(input, residual, residual, nullptr, weight, scale_tensor, output, next_buffer, epsilon, cols,
                                                           buffer_cols);
}

// For the MLP block (residual_rms_into): at most 64 rows, so nothing is read past the caches.
template <int DT, int ITERS>
__global__ void __launch_bounds__(kRmsMaxThreads) residual_rms_into_kernel(
    const uint16_t* input, const uint16_t* residual_in, uint16_t* residual, uint16_t* input_copy, const uint16_t* __restrict__ weight,
    const float* __restrict__ scale_tensor, void* __restrict__ output, float epsilon, int cols) {
    residual_rms_vec<DT, true, ITERS, false, true>(input, residual_in, residual, input_copy, weight, scale_tensor, output, nullptr, epsilon, cols, 0);
}

// One element per thread per iteration; no alignment or divisibility requirement.  The second pass re-reads the
// residual this same thread wrote in the first.
template <int DT, bool FP8_OUT>
__global__ void __launch_bounds__(kRmsMaxThreads) residual_rms_scalar_kernel(
    const uint16_t* __restrict__ input, uint16_t* __restrict__ residual, const uint16_t* __restrict__ weight,
    const float* __restrict__ scale_tensor, void* __restrict__ output, uint16_t* __restrict__ next_buffer,
    float epsilon, int cols, int buffer_cols) {
    __shared__ __align__(16) float red[16];
    const long row_off = (long)blockIdx.x * cols;
    float ssq = 0.f;
    for (int i = threadIdx.x; i < cols; i += blockDim.x) {
        const uint16_t z = store16<DT>(load16<DT>(input[row_off + i]) + load16<DT>(residual[row_off + i]));
        const float f = load16<DT>(z);
        ssq += f * f;
        residual[row_off + i] = z;
    }
    const float total = block_sum(ssq, red);
    const float norm = rsqrtf(total / (float)cols + epsilon);
    float inv_scale = 1.f;
    if constexpr (FP8_OUT) inv_scale = 1.f / scale_tensor[0];
    for (int i = threadIdx.x; i < cols; i += blockDim.x) {
        const float zf = load16<DT>(residual[row_off + i]);
        const float wf = load16<DT>(weight[i]);
        if constexpr (FP8_OUT) {
            static_cast<uint8_t*>(output)[row_off + i] = cvt_fp8(zf * norm * wf * inv_scale);
        } else {
            const uint16_t n16 = store16<DT>(zf * norm);
            static_cast<uint16_t*>(output)[row_off + i] = store16<DT>(load16<DT>(n16) * wf);
        }
    }
    zero_next_buffer_row(next_buffer, buffer_cols);
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// threads per row of nvec 16-byte pieces: enough for one or two each, whole wavefronts, at most 1024
static int rms_threads(int nvec) {
    int threads = ((nvec + 63) / 64) * 64;
    if (threads > 512) threads = ((nvec + 127) / 128) * 64;
    if (threads > kRmsMaxThreads) threads = kRmsMaxThreads;
    return threads < 64 ? 64 : threads;
}

template <int DT, bool FP8_OUT>
static int launch_rms(const void* input, void* residual, const void* weight, const float* scale_tensor, float epsilon,
                      void* output, void* next_buffer, int rows, int cols, int buffer_cols, int num_threads,
                      bool force_scalar, hipStream_t stream) {
    const uint16_t* in = static_cast<const uint16_t*>(input);
    uint16_t* res = static_cast<uint16_t*>(residual);
    const uint16_t* w = static_cast<const uint16_t*>(weight);
    uint16_t* nb = static_cast<uint16_t*>(next_buffer);
    // 16-byte path: aligned rows (cols % 8 == 0 keeps every row aligned) and an aligned output row
    const bool out_ok = FP8_OUT ? ((reinterpret_cast<uintptr_t>(output) & 7) == 0) : aligned16(output);
    bool vec = !force_scalar && (cols % 8 == 0) && aligned16(input) && aligned16(residual) && aligned16(weight) && out_ok;
    int threads = num_threads;
    if (vec) {
        const int nvec = cols / 8;
        if (threads == 0) threads = rms_threads(nvec);
        const int iters = (nvec + threads - 1) / threads;
        if (iters > 4) vec = false;  // would not fit the register cache: fall through to the strided kernel
        else {
#define HFRK_RMS_LAUNCH(IT, ONCE)                                                                                          \
    hipLaunchKernelGGL((residual_rms_vec_kernel<DT, FP8_OUT, IT, ONCE>), dim3(rows), dim3(threads), 0, stream, in, res, w, \
                       scale_tensor, output, nb, epsilon, cols, buffer_cols)
#define HFRK_RMS_ITERS(ONCE)                         \
    do {                                             \
        if (iters <= 1) HFRK_RMS_LAUNCH(1, ONCE);    \
        else if (iters == 2) HFRK_RMS_LAUNCH(2, ONCE); \
        else HFRK_RMS_LAUNCH(4, ONCE);               \
    } while (0)
            if ((long)rows * cols >= kReadOnceFrom) HFRK_RMS_ITERS(true);
            else HFRK_RMS_ITERS(false);
#undef HFRK_RMS_ITERS
#undef HFRK_RMS_LAUNCH
        }
    }
    if (!vec) {
        if (threads == 0) {
            threads = ((cols + 63) / 64) * 64;
            if (threads > kRmsMaxThreads) threads = kRmsMaxThreads;
        }
        hipLaunchKernelGGL((residual_rms_scalar_kernel<DT, FP8_OUT>), dim3(rows), dim3(threads), 0, stream, in, res, w,
                           scale_tensor, output, nb, epsilon, cols, buffer_cols);
    }
    HFRK_HIP_TRY(hipGetLastError());
    return HFRK_SUCCESS;
}

bool residual_rms_into_takes(const void* input, const void* residual_in, const void* residual, const void* input_copy, const void* weight, const void* output,
                             int cols) {
    return cols % 8 == 0 && cols <= 4 * 8 * kRmsMaxThreads && aligned16(input) && aligned16(residual_in) && aligned16(residual) && aligned16(input_copy) &&
           aligned16(weight) && (reinterpret_cast<uintptr_t>(output) & 7) == 0;
}

template <int DT>
static int launch_rms_into(const void* input, const void* residual_in, void* residual, void* input_copy, const void* weight, const float* scale_tensor,
                           float epsilon, void* output, int rows, int cols, hipStream_t stream) {
    const int threads = rms_threads(cols / 8), iters = (cols / 8 + threads - 1) / threads;
#define HFRK_RMS_LAUNCH(IT)                                                                                                         \
    hipLaunchKernelGGL((residual_rms_into_kernel<DT, IT>), dim3(rows), dim3(threads), 0, stream, static_cast<const uint16_t*>(input), \
                       static_cast<const uint16_t*>(residual_in), static_cast<uint16_t*>(residual), static_cast<uint16_t*>(input_copy), \
                       static_cast<const uint16_t*>(weight), scale_tensor, output, epsilon, cols)
    if (iters <= 1) HFRK_RMS_LAUNCH(1);
    else if (iters == 2) HFRK_RMS_LAUNCH(2);
    else HFRK_RMS_LAUNCH(4);
#undef HFRK_RMS_LAUNCH
    HFRK_HIP_TRY(hipGetLastError());
    return HFRK_SUCCESS;
}

int residual_rms_into(const void* input, const void* residual_in, void* residual, void* input_copy, const void* weight, const float* scale_tensor,
                      float epsilon, void* output, int rows, int cols, int io_dtype, hipStream_t stream) {
    if (!residual_rms_into_takes(input, residual_in, residual, input_copy, weight, output, cols)) return HFRK_BAD_ALIGNMENT;
    return io_dtype == HFRK_F16 ? launch_rms_into<HFRK_F16>(input, residual_in, residual, input_copy, weight, scale_tensor, epsilon, output, rows, cols, stream)
                                : launch_rms_into<HFRK_BF16>(input, residual_in, residual, input_copy, weight, scale_tensor, epsilon, output, rows, cols, stream);
}

}  // namespace hfrk

extern "C" int hfrk_residual_rms(const void* input, void* residual, const void* weight, const float* scale_tensor,
                                 float epsilon, void* output, void* next_buffer, int rows, int cols, int buffer_cols,
                                 int io_dtype, int out_dtype, int num_threads, int force_scalar, void* stream) {
    using namespace hfrk;
    if (rows < 0 || cols < 1 || buffer_cols < 0) return HFRK_BAD_SHAPE;
    if (rows == 0) return HFRK_SUCCESS;
    if (!input || !residual || !weight || !output) return HFRK_BAD_SHAPE;
    if (buffer_cols > 0 && !next_buffer) return HFRK_BAD_SHAPE;
    if (io_dtype != HFRK_F16 && io_dtype != HFRK_BF16) return HFRK_BAD_DTYPE;
    if (out_dtype != HFRK_FP8_E4M3FN && out_dtype != io_dtype) return HFRK_BAD_DTYPE;
    if (out_dtype == HFRK_FP8_E4M3FN && !scale_tensor) return HFRK_BAD_SHAPE;
    if (num_threads < 0 || num_threads > kRmsMaxThreads || (num_threads % 64) != 0) return HFRK_INVALID_CONFIG;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool fs = force_scalar != 0;
    const bool fp8 = out_dtype == HFRK_FP8_E4M3FN;
    if (io_dtype == HFRK_F16) {
        return fp8 ? launch_rms<HFRK_F16, true>(input, residual, weight, scale_tensor, epsilon, output, next_buffer, rows, cols, buffer_cols, num_threads, fs, s)
                   : launch_rms<HFRK_F16, false>(input, residual, weight, scale_tensor, epsilon, output, next_buffer, rows, cols, buffer_cols, num_threads, fs, s);
    }
    return fp8 ? launch_rms<HFRK_BF16, true>(input, residual, weight, scale_tensor, epsilon, output, next_buffer, rows, cols, buffer_cols, num_threads, fs, s)
               : launch_rms<HFRK_BF16, false>(input, residual, weight, scale_tensor, epsilon, output, next_buffer, rows, cols, buffer_cols, num_threads, fs, s);
}
