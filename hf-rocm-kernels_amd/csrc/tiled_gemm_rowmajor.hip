// Tiled GEMM on row-major weights (tiled_gemm_kernel.h).
#include "tiled_gemm_kernel.h"

namespace hfrk {

// The 256 x 128 tile's number of waves.  Eight, unless rows of A or B begin inside a 128-byte line (k or the weight's stride no multiple of
// it): a stage of such a row lies across two lines, and eight waves lose more by that than four (us, eight / four waves, weights out of the caches:
// 512 x 10240 x 8192 57.7 / 57.8, with a stride of 8256 64.3 / 58.5, k = 8256 77.3 / 66.7, k = 8208 81.7 / 74.0; 496 x 9840 x 10688 99.1 / 81.5;
// 220 x 23912 x 8928 91.5 / 81.0; in layer calls on one weight, which the 256 MB cache holds from pass to pass, 496 x 9840 x 10688 104.8 / 87.8,
// 471 x 12432 x 5872 64.9 / 59.1, 2010 x 3288 x 16992 138.5 / 140.2, 721 x 9408 x 4160 39.1 / 40.2).  A last row of tiles less than half full brings weight lines into L2 ahead of its neighbours, and does it
// better on eight (300 x 6144 x 8256 50.0 / 55.3, 560 x 28672 x 4112 100 / 104, 784 x 10240 x 4160 59.2 / 63.8; even at half: 384 x 6144 x
// 8256 58.3 / 57.4, 640 x 10240 x 4160 36.9 / 38.2) as long as it is one of up to four, or the workgroups are few (2404 x 2056 x 2096
// 20.3 / 21.5, 1320 x 6144 x 8256 116.2 / 120.4; but 1040 x 12432 x 5872 107.1 / 101.9, 1347 x 24256 x 8368 361 / 346).
static bool four_waves(const TiledGemmArgs& a) {
    if (((a.k | a.b_stride) & 127) == 0) return false;
    const int last_rows = a.m - (a.tiles_m - 1) * kTiledShapes[1].bm;
    return 2 * last_rows >= kTiledShapes[1].bm || (a.tiles_m > 4 && 2 * a.tiles_m * a.tiles_n * a.splits > 3 * kNumCU);
}

int launch_tiled_rowmajor(const TiledGemmArgs& args, int shape, hipStream_t stream) {
    if (shape == 1 && four_waves(args)) {
#define HFRK_TILED_LAUNCH(I, TM, TN, WM, WN, NST, WGS) \
    return launch_tiled_shape<TM, TN, WM, WN, NST, WGS, false>(args, tiled_lds_bytes(kTiledShapes[I]), stream);
        HFRK_TILED_FOUR_WAVES(HFRK_TILED_LAUNCH)
#undef HFRK_TILED_LAUNCH
    }
    return launch_tiled<false>(args, shape, stream);
}

}  // namespace hfrk
