// Tiled GEMM on weights in the packed load format (tiled_gemm_kernel.h).
#include "tiled_gemm_kernel.h"

namespace hfrk {
int launch_tiled_packed(const TiledGemmArgs& args, int shape, hipStream_t stream) { return launch_tiled<true>(args, shape, stream); }
}  // namespace hfrk
