// Tiled GEMM on row-major weights (tiled_gemm_kernel.h).
#include "tiled_gemm_kernel.h"

namespace hfrk {

// The 256 x 128 tile's number of waves: eight, unless rows of A or B begin inside a 128-byte line (k or the weight's stride no multiple of it) and
// a workgroup's k is long.  A stage of such a row lies across two lines, and where the weight comes from memory eight waves lose more by that than
// four (us, eight / four: 512 x 10240 x 8192 57.7 / 57.8, with a stride of 8256 64.3 / 58.5, k = 8256 77.3 / 66.7; 496 x 9840 x 10688 99.1 / 81.5,
// 1223 x 4752 x 21584 193 / 164); prologue and epilogue are the cheaper on eight.  75 drawn sizes whose plan is this tile: from 44 stages per
// workgroup on and k in one or two parts four waves are 9 % faster in the mean (0 to 18 %) and level on a weight that the 256 MB cache holds from
// call to call (6 % slower, 2208 x 2432 x 8256, to 13 % faster; 194 x 14688 x 14448, which just fits, 12 % slower in one run and 9 % faster in
// another); on the others 3 % faster from memory and 5 % slower from the cache.
// A last row of tiles that is less than about half full brings weight lines into L2 ahead of its neighbours, and does it better on eight
// (300 x 6144 x 8256 50.0 / 55.3, 384 x 6144 x 8256 58.3 / 57.4, 300 x 28672 x 8256 114 / 122), as long as it is one of up to four or the
// workgroups are few (1320 x 6144 x 8256 116.2 / 120.4; but 1040 x 12432 x 5872 107.1 / 101.9, 1347 x 24256 x 8368 361 / 346).
static bool four_waves(const TiledGemmArgs& a) {
    if (((a.k | a.b_stride) & 127) == 0 || a.stages_q < 44 || a.splits > 2) return false;
    const int last_rows = a.m - (a.tiles_m - 1) * kTiledShapes[1].bm;
    return 16 * last_rows >= 9 * kTiledShapes[1].bm || (a.tiles_m > 4 && 2 * a.tiles_m * a.tiles_n * a.splits > 3 * kNumCU);
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
