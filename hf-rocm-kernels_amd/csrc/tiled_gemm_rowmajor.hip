// Tiled GEMM on row-major weights (tiled_gemm_kernel.h).
#include "tiled_gemm_kernel.h"

namespace hfrk {
int launch_tiled_rowmajor(const TiledGemmArgs& args, int shape, hipStream_t stream) { return launch_tiled<false>(args, shape, stream); }
}  // namespace hfrk
