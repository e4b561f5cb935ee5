// output[r,c] = e4m3fn( clamp( silu(gate_up[r,c]) * gate_up[r,cols+c] / scale, +-448 ) );  next_buffer <- 0
//
// Replaces csrc/op_src/swiglu/swiglu_dispatch.cu:8-42 and its kernels (swiglu_scalar.cu:24-66,
// swiglu_vectorized.cu:27-97).  Pure streaming op: 16-byte loads of 8 gate and 8 up values, fp32 math
// (x * 1/(1 + 2^(-x*log2 e)), the same exp2 form as the reference), one 8-byte store of 8 fp8 values.
// The clamp is +-448, the largest e4m3fn value (the reference's vectorised kernel clamps at 224 because its
// fnuz encoding tops out at 240, csrc/utils/macros.h:15).
#include "hfrk_internal.h"

namespace hfrk {

// Zero rows*buffer_cols 16-bit elements, spread over every thread of the grid.
__device__ __forceinline__ void zero_next_buffer(uint16_t* next_buffer, long total) {
    if (total <= 0) return;
    const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long nthreads = (long)gridDim.x * blockDim.x;
    const uintptr_t addr = reinterpret_cast<uintptr_t>(next_buffer);
    long head = (long)(((16 - (addr & 15)) & 15) >> 1);
    if (head > total) head = total;
    const long body = (total - head) >> 3;
    for (long i = tid; i < head; i += nthreads) next_buffer[i] = 0;
    uint4* const vec = reinterpret_cast<uint4*>(next_buffer + head);
    for (long i = tid; i < body; i += nthreads) vec[i] = make_uint4(0, 0, 0, 0);
    for (long i = head + body * 8 + tid; i < total; i += nthreads) next_buffer[i] = 0;
}

constexpr int kSwigluPieces = 2;

// Bound by memory.  A thread requests all its pieces before it works on the first, and each further set behind them.  INDEX is
// 32 bits wide wherever the pieces can be counted in it: the division by the row length is per piece, and in 64 bits it was most
// of the kernel's instructions.  fp16, us, before both / now: 2048 x 6656 13.8 / 12.6, the same buffers again and again (136 MB, in the
// caches) 12.3 / 11.05; 256 x 14336 4.9 / 4.6.
// TOGETHER: a workgroup's pieces follow one another; otherwise a thread's are a whole launch apart.  Apart is faster up to about 3.5
// million pieces (2048 x 6656 12.3 / 12.6 together, 1228 x 8384 9.25 / 9.55), together from 4 million on (kTogetherFrom: 4096 x 8192
// 28.9 / 28.5, 3408 x 14520 40.6 / 39.7, and 4007 x 8272, where the two halves fall on the same channels, 31.7 / 29.5).
constexpr long kTogetherFrom = 4000000;

template <int DT, typename INDEX, bool TOGETHER>
__global__ void __launch_bounds__(1024) swiglu_vec_kernel(const uint16_t* __restrict__ gate_up,
                                                          const float* __restrict__ scale_tensor,
                                                          uint8_t* __restrict__ output, uint16_t* __restrict__ next_buffer,
                                                          int rows, int cols, int buffer_cols) {
    const INDEX vpr = (INDEX)(cols >> 3);  // 8-element pieces per output row
    const INDEX nvec = (INDEX)rows * vpr;
    const INDEX launch = (INDEX)gridDim.x * blockDim.x;
    const INDEX stride = TOGETHER ? (INDEX)blockDim.x : launch;  // between a thread's pieces
    const INDEX first = (INDEX)blockIdx.x * (TOGETHER ? kSwigluPieces : 1) * blockDim.x + threadIdx.x;
    v4i g[kSwigluPieces], u[kSwigluPieces];
    auto fetch = [&](INDEX at) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < kSwigluPieces; ++p) {
            const INDEX v = at + p * stride;
            if (v < nvec) {
                const INDEX r = v / vpr;
                const uint16_t* const grow = gate_up + (long)r * 2 * cols;
                g[p] = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(grow) + (v - r * vpr));
                u[p] = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(grow + cols) + (v - r * vpr));
            }
        }
    };
    fetch(first);
    const float s = scale_tensor[0];
    const float inv_scale = (s != 0.f) ? 1.f / s : 1.f;
    for (INDEX at = first; at < nvec; at += kSwigluPieces * launch) {
        if (at != first) fetch(at);
#pragma unroll
        for (int p = 0; p < kSwigluPieces; ++p) {
            const INDEX v = at + p * stride;
            if (v >= nvec) break;
            float y[8];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t gw = (uint32_t)g[p][j], uw = (uint32_t)u[p][j];
                y[2 * j] = silu_mul(load16<DT>((uint16_t)(gw & 0xffff)), load16<DT>((uint16_t)(uw & 0xffff)), inv_scale);
                y[2 * j + 1] = silu_mul(load16<DT>((uint16_t)(gw >> 16)), load16<DT>((uint16_t)(uw >> 16)), inv_scale);
            }
            uint32_t p0 = cvt_pk_fp8(y[0], y[1], 0u, false);
            p0 = cvt_pk_fp8(y[2], y[3], p0, true);
            uint32_t p1 = cvt_pk_fp8(y[4], y[5], 0u, false);
            p1 = cvt_pk_fp8(y[6], y[7], p1, true);
            // rows of the output follow one another: piece v lies at 8 v
            reinterpret_cast<uint2*>(output)[v] = make_uint2(p0, p1);
        }
    }
    zero_next_buffer(next_buffer, (long)rows * buffer_cols);
}

template <int DT>
__global__ void __launch_bounds__(1024) swiglu_scalar_kernel(const uint16_t* __restrict__ gate_up,
                                                             const float* __restrict__ scale_tensor,
                                                             uint8_t* __restrict__ output, uint16_t* __restrict__ next_buffer,
                                                             int rows, int cols, int buffer_cols) {
    const long total = (long)rows * cols;
    const float s = scale_tensor[0];
    const float inv_scale = (s != 0.f) ? 1.f / s : 1.f;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
        const long r = i / cols;
        const int c = (int)(i - r * cols);
        const float g = load16<DT>(gate_up[r * 2 * cols + c]);
        const float u = load16<DT>(gate_up[r * 2 * cols + cols + c]);
        output[i] = cvt_fp8(silu_mul(g, u, inv_scale));
    }
    zero_next_buffer(next_buffer, (long)rows * buffer_cols);
}

}  // namespace hfrk

extern "C" int hfrk_swiglu(const void* gate_up, const float* scale_tensor, void* output, void* next_buffer, int rows,
                           int cols, int buffer_cols, int io_dtype, int num_threads, int force_scalar, void* stream) {
    using namespace hfrk;
    if (rows < 0 || cols < 1 || buffer_cols < 0) return HFRK_BAD_SHAPE;
    if (rows == 0) return HFRK_SUCCESS;
    if (!gate_up || !scale_tensor || !output) return HFRK_BAD_SHAPE;
    if (buffer_cols > 0 && !next_buffer) return HFRK_BAD_SHAPE;
    if (io_dtype != HFRK_F16 && io_dtype != HFRK_BF16) return HFRK_BAD_DTYPE;
    if (num_threads < 0 || num_threads > 1024) return HFRK_INVALID_CONFIG;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const uint16_t* in = static_cast<const uint16_t*>(gate_up);
    uint8_t* out = static_cast<uint8_t*>(output);
    uint16_t* nb = static_cast<uint16_t*>(next_buffer);
    const bool vec = !force_scalar && (cols % 8 == 0) && (reinterpret_cast<uintptr_t>(gate_up) & 15) == 0 &&
                     (reinterpret_cast<uintptr_t>(output) & 7) == 0;
    int threads = num_threads > 0 ? num_threads : 256;
    const long work = vec ? (long)rows * (cols / 8) : (long)rows * cols;
    long blocks = (work + threads - 1) / threads;
    // one piece per thread until the chip is full of threads (2048 per compute unit), then kSwigluPieces; the loop in the kernel
    // strides over what a launch of 64 workgroups per compute unit leaves
    if (vec && work > (long)kNumCU * 2048) blocks = (work + (long)threads * kSwigluPieces - 1) / ((long)threads * kSwigluPieces);
    const long cap = vec ? (long)kNumCU * 64 : (long)kNumCU * 16;
    if (blocks > cap) blocks = cap;
    if (blocks < 1) blocks = 1;
    // no index of a thread, the first one past the end among them, leaves 32 bits
    const bool narrow = work + 2L * kSwigluPieces * blocks * threads < (1L << 32);
#define HFRK_SWIGLU(KERNEL) \
    hipLaunchKernelGGL((KERNEL), dim3((unsigned)blocks), dim3(threads), 0, s, in, scale_tensor, out, nb, rows, cols, buffer_cols)
#define HFRK_SWIGLU_VEC(DT_)                                                        \
    do {                                                                            \
        if (!narrow) HFRK_SWIGLU((swiglu_vec_kernel<DT_, uint64_t, true>));         \
        else if (work >= kTogetherFrom) HFRK_SWIGLU((swiglu_vec_kernel<DT_, uint32_t, true>)); \
        else HFRK_SWIGLU((swiglu_vec_kernel<DT_, uint32_t, false>));                \
    } while (0)
    if (io_dtype == HFRK_F16) {
        if (!vec) HFRK_SWIGLU(swiglu_scalar_kernel<HFRK_F16>);
        else HFRK_SWIGLU_VEC(HFRK_F16);
    } else {
        if (!vec) HFRK_SWIGLU(swiglu_scalar_kernel<HFRK_BF16>);
        else HFRK_SWIGLU_VEC(HFRK_BF16);
    }
#undef HFRK_SWIGLU_VEC
#undef HFRK_SWIGLU
    HFRK_HIP_TRY(hipGetLastError());
    return HFRK_SUCCESS;
}
