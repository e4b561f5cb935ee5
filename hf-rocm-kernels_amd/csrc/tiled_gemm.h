// Launch arguments and tile shapes of the tiled GEMM (calls with more rows than the skinny kernels take).
#pragma once

#include "skinny_gemm_args.h"

#include <type_traits>

namespace hfrk {

struct TiledGemmArgs {
    const uint8_t* A;
    const uint8_t* B;
    void* D;
    const void* base;  // 16-bit addend or null
    int base_stride;   // elements between its rows; 0: one row for all (a bias)
    const float* scale_a;
    const float* scale_b;
    int sa_stride, sb_stride;
    int m, n, k, b_stride;
    int d_dtype;
    int vec;                      // rows of D and base are 16-byte aligned
    int tiles_m, tiles_n, group_m;
    int stages_q, stages_r;       // k stages per split, the first stages_r splits one more
    int splits;
    int window, phase_m, phase_n;  // stages within which a workgroup's start in k is turned; 65536ths of a turn per row and column of tiles
    float* ws;
    uint32_t ws_bytes;
    int* counters;
};

constexpr int kTiledStage = 128;    // bytes of k per pipeline stage

// TM x TN matrix tiles of 32 x 32 per wave, WM x WN waves, NST stages (or halves of them) of operands in LDS, WGS workgroups per compute unit.
// X(index, TM, TN, WM, WN, NST, WGS)
#define HFRK_TILED_SHAPES(X) \
    X(0, 4, 2, 2, 4, 5, 1)   \
    X(1, 2, 2, 4, 2, 3, 1)   \
    X(2, 2, 2, 2, 2, 5, 1)   \
    X(3, 2, 1, 2, 2, 3, 2)   \
    X(4, 1, 1, 2, 2, 8, 1)
// Shape 1 on four waves, for row-major operands whose rows begin inside a 128-byte line and a long k (tiled_gemm_rowmajor.hip).
#define HFRK_TILED_FOUR_WAVES(X) X(1, 4, 2, 2, 2, 3, 1)

// The shapes whose multiplying waves load for themselves where a workgroup's k is one or two stages.  Waves that only load have nothing to run ahead
// of there, and starting them costs: over 285 sizes of one stage and 274 of two on 128 x 64 tiles 3.5 and 1.7 % (165 x 9040 x 512 packed 6.9 us without, 7.7
// with them), on eight of the 256 x 128 tile 3 %; from three stages on the two are level, from eight on they win.
#define HFRK_TILED_SHORT_K(X) \
    X(1, 2, 2, 4, 2, 3, 1)    \
    X(3, 2, 1, 2, 2, 3, 2)

// Whether LDS holds halves of stages (the 256 x 256 tile: five halves, 160 KB; two whole stages are 128).
constexpr bool tiled_half_stages(int tm, int waves) { return tm * waves >= 32; }
// Waves of a workgroup that only load, beside the WM x WN that multiply (tiled_gemm_kernel.h).
constexpr int tiled_loader_waves(int tm) { return tm < 4 ? 4 : 0; }

struct TiledShape {
    int bm, bn, stages, per_cu;
    bool halves;
    int threads;  // per workgroup, at most
};
#define HFRK_TILED_ROW(I, TM, TN, WM, WN, NST, WGS) {32 * TM * WM, 32 * TN * WN, NST, WGS, tiled_half_stages(TM, WM * WN), 64 * (WM * WN + tiled_loader_waves(TM))},
constexpr TiledShape kTiledShapes[] = {HFRK_TILED_SHAPES(HFRK_TILED_ROW)};
#undef HFRK_TILED_ROW
#define HFRK_TILED_SAME(I, TM, TN, WM, WN, NST, WGS) \
    static_assert(kTiledShapes[I].bm == 32 * TM * WM && kTiledShapes[I].bn == 32 * TN * WN && kTiledShapes[I].stages == NST && kTiledShapes[I].per_cu == WGS);
HFRK_TILED_FOUR_WAVES(HFRK_TILED_SAME)
HFRK_TILED_SHORT_K(HFRK_TILED_SAME)
#undef HFRK_TILED_SAME
constexpr int kTiledShapeCount = sizeof(kTiledShapes) / sizeof(kTiledShapes[0]);
constexpr int tiled_lds_bytes(const TiledShape& s) { return (s.bm + s.bn) * (s.halves ? kTiledStage / 2 : kTiledStage) * s.stages; }

// tiled_gemm.hip
bool tiled_size_ok(int m, int n, int k);
// Whether the tiled GEMM is the faster one for a call that the skinny GEMM would run under `skinny`, and the plan it then takes.
bool tiled_instead(int m, int n, int k, const hfrk_gemm_plan& skinny, hfrk_tiled_plan* plan);
size_t tiled_plan_ws_bytes(const hfrk_tiled_plan& p, int m, int n);
long tiled_plan_counters(const hfrk_tiled_plan& p, int m, int n);
// The launch alone: arguments are checked and the plan fits them and the workspace.
int tiled_launch(const void* A, const void* B, bool packed, void* D, const void* base, int base_stride, const float* scale_a, int sa_stride,
                 const float* scale_b, int sb_stride, int m, int n, int k, int b_stride, int d_dtype, const hfrk_tiled_plan& p, float* ws, size_t ws_bytes,
                 int* counters, hipStream_t stream);
int launch_tiled_rowmajor(const TiledGemmArgs& args, int shape, hipStream_t stream);  // tiled_gemm_rowmajor.hip
int launch_tiled_packed(const TiledGemmArgs& args, int shape, hipStream_t stream);    // tiled_gemm_packed.hip

}  // namespace hfrk
