// Host side of the tiled GEMM: plan and entry points (the kernel is in tiled_gemm_kernel.h).
#include <math.h>

#include "tiled_gemm.h"

namespace hfrk {

static int div_up(long a, long b) { return (int)((a + b - 1) / b); }

bool tiled_size_ok(int m, int n, int k) {
    // every offset the kernel forms inside one tile's buffers stays below 2^31, every tile count and workspace index in 32 bits
    constexpr int kMost = 1 << 21;
    return m >= 1 && n >= 1 && k >= 1 && m <= (1 << 24) && n <= kMost && k <= kMost &&
           (long)div_up(m, 64) * div_up(n, 64) < (1L << 24);
}

static size_t tiled_ws_bytes(const TiledShape& s, int m, int n, int splits) {
    return splits <= 1 ? 0 : (size_t)div_up(m, s.bm) * div_up(n, s.bn) * splits * s.bm * s.bn * sizeof(float);
}

size_t tiled_plan_ws_bytes(const hfrk_tiled_plan& p, int m, int n) { return tiled_ws_bytes(kTiledShapes[p.shape], m, n, p.splits); }
long tiled_plan_counters(const hfrk_tiled_plan& p, int m, int n) {
    const TiledShape& s = kTiledShapes[p.shape];
    return p.splits <= 1 ? 0 : (long)div_up(m, s.bm) * div_up(n, s.bn);
}

static int check_tiled_plan(int m, int n, int k, const hfrk_tiled_plan& p) {
    if (p.shape < 0 || p.shape >= kTiledShapeCount || p.splits < 1 || p.group_m < 1) return HFRK_INVALID_CONFIG;
    const TiledShape& s = kTiledShapes[p.shape];
    const long tiles = (long)div_up(m, s.bm) * div_up(n, s.bn);
    if (p.splits > div_up(k, kTiledStage) || p.group_m > div_up(m, s.bm)) return HFRK_INVALID_CONFIG;
    if (p.splits > 1 && (tiled_ws_bytes(s, m, n, p.splits) > kWsFloats * sizeof(float) || tiles > kMaxPanels)) return HFRK_INVALID_CONFIG;
    return HFRK_SUCCESS;
}

// The shape and the number of k splits with the smallest predicted time, in us.  The constants are fitted to a sweep so that the choices come
// out right (profiles/tiled_gemm_plans.csv: 260 sizes, 3640 calls, row-major weights rotated through 768 MB, k whole stages; on four sizes the
// choice is a split that the sweep does not have): the choice is 0.25 % slower than the best measured plan in the geometric mean, 5 % or
// more on 6 sizes, 14 % on the worst (613 x 23408 x 3584 90 us instead of 79, with 782 x 16888 x 3584 8 % the same: 128 x 128 where 256 x 128
// is faster); on every third size, with the others fitted, 0.4 %, and with the quantisation kernel in front of each call 0.2 %.  Against the
// constants before, which were for these tiles on four waves, 54 choices differ, 10 % faster in the mean; one is 6 % slower.  On 73 drawn sizes
// where the two differ the choices are 9 % faster in the mean on weights from memory, and 1.5 % on one weight that the 256 MB cache holds from call
// to call; there 12 of them are 7 to 23 % slower, most of them splits of a long k (722 x 2000 x 16384 33.7 / 41.3 us, from memory 40.5 / 40.6).
// Terms for the operands' traffic out of L2 and for the weight's out of memory came out idle.  The sweep was timed before the tiles had waves that
// only load and stages by halves; with them, on 396 drawn sizes of 65 to 4096 rows, the choices are 0.7 % slower than the best plan in the mean.
static float tiled_cost(int m, int n, int k, int shape, int splits) {
    struct Shape { float fixed, stage; };  // a workgroup's prologue and epilogue; one stage of 128 bytes of k
    static constexpr Shape kShape[kTiledShapeCount] = {{8.81f, 1.28f}, {8.88f, .643f}, {5.10f, .491f}, {2.97f, .398f}, {3.53f, .240f}};
    constexpr float kShares = 6.41e6f;                       // bytes per us of partial sums
    constexpr float kPairFixed = 1.29f, kPairStage = 1.61f;  // two workgroups on a compute unit against one
    const TiledShape& s = kTiledShapes[shape];
    const long wgs = (long)div_up(m, s.bm) * div_up(n, s.bn) * splits, slots = (long)kNumCU * s.per_cu;
    const float stages = (float)div_up(k, kTiledStage) / splits;
    auto round_us = [&](long count) {
        if (count == 0) return 0.f;
        const bool pair = count > kNumCU;
        return kShape[shape].fixed * (pair ? kPairFixed : 1.f) + stages * kShape[shape].stage * (pair ? kPairStage : 1.f);
    };
    float t = (float)(wgs / slots) * round_us(slots) + round_us(wgs % slots);
    if (splits > 1) t += .451f + .797f * splits + (float)wgs * s.bm * s.bn * 8.f / kShares;
    return t;
}

constexpr int kTiledMaxSplits = 8;

// Up to 64 rows: one row of tiles streams the weight.  64 x 64 tiles with k in up to 8 parts of 4 stages or more on at most 512 workgroups, or,
// where they take a second round, 128 x 64 tiles, two on a compute unit.  In us, the constants fitted to 1300 sizes of 17 to 64 rows with weights from
// memory (5300 calls; median error 2.7 %, 90 % of them within 8 %); weights that the 256 MB cache holds are up to 45 % faster.
static float few_rows_cost(int m, int n, int k, int shape, int splits) {
    struct Shape { float fixed, stage, rows, bytes_per_us, start, overlap; };
    static constexpr Shape kWide = {3.15f, .334f, .204f, 7.82e6f, 3.97f, .501f}, kNarrow = {2.31f, .0566f, .209f, 8.74e6f, 3.08f, .469f};
    const Shape& c = shape == 3 ? kWide : kNarrow;
    const long wgs = (long)div_up(n, 64) * splits;
    const int rounds = shape == 3 ? 1 : div_up(wgs, kNumCU);
    const float work = rounds * (c.fixed + (float)div_up(k, kTiledStage) / splits * (c.stage + c.rows * (m + 64) / 128.f));
    const float stream = (float)n * k / c.bytes_per_us + c.start;
    float t = fmaxf(work, stream) + c.overlap * fminf(work, stream);
    if (splits > 1) t += .552f + .335f * splits + 1.859f * wgs / kNumCU;
    return t;
}

// The fit's sizes have k in whole stages.  Rows of another k begin inside a 128-byte line, and from memory the fit then takes too few parts of it: up
// to four of 8 stages or more are kept where a compute unit each has room for them (62 x 8096 x 3088 in two parts 13.3 us, in one 16.6; 55 x 3920 x 6416 in four
// 13.9, in three 15.3; of 814 drawn sizes of 33 to 64 rows 30 had fewer, 7 % slower from memory and 12 % faster from the cache).  Below 13 stages it
// takes two or three for nothing (54 x 192 x 1344 6.14 us in one, 6.64 in two; 17 sizes, 4 % slower from the cache, 1 % faster from memory).
static float make_few_rows_plan(int m, int n, int k, int max_splits, hfrk_tiled_plan* plan) {
    const int stages = div_up(k, kTiledStage);
    const long tiles = div_up(n, 64);
    int least = 1;
    if (k % 256 != 0) {
        for (least = 4; least > 1 && (least > max_splits || least * tiles > kNumCU || least * 8 > stages);) --least;
        if (stages < 13) max_splits = 1;
    }
    float best = INFINITY;
    auto offer = [&](int shape, int splits) {
        const float t = few_rows_cost(m, n, k, shape, splits);
        if (t < .99f * best) {  // of equals the one with the fewest parts
            best = t;
            *plan = {shape, splits, 1};
        }
    };
    if (least == 1) offer(4, 1);
    if (tiles > kNumCU && tiles <= 2 * kNumCU) offer(3, 1);
    for (int splits = least < 2 ? 2 : least; splits <= max_splits && 4 * splits <= stages && tiles * splits <= 2 * kNumCU; ++splits) offer(4, splits);
    return best;
}

// What the workgroup kernel (skinny_gemm.hip) takes under a plan of its own, in us: its unit is a panel's rows and a slab of k, workgroups that
// share a panel exchange their sums.  Fitted to 1079 of the same calls by the number of waves along k (median error 6 %, 90 % of them within 12 to 18 %).
static float workgroup_kernel_cost(int m, int n, int k, const hfrk_gemm_plan& p) {
    struct Waves { float fixed, bytes, rows, bytes_per_us, overlap, exchange, share; };
    static constexpr Waves kWaves[3] = {{3.45f, .000869f, 36.8f, 19.1e6f, 2.53f, 4.98f, .0073f},
                                        {3.72f, .00150f, 15.1f, 8.94e6f, .968f, 3.65f, .0124f},
                                        {4.87f, .00162f, 19.7f, 5.85e6f, 0.f, 1.01f, .0516f}};
    const Waves& c = kWaves[p.wk >= 4 ? 2 : p.wk - 1];
    const long units = (long)p.panels * p.slabs, per = units / p.grid;
    const int padded = 16 * div_up(m, 16);
    const float work = (float)div_up(units, p.grid) * c.bytes * (16 * p.wn + c.rows * padded) * (p.wk * p.ch) * .25f;
    const float stream = (float)n * k / c.bytes_per_us;
    float t = c.fixed + fmaxf(work, stream) + c.overlap * fminf(work, stream);
    if (p.panels % p.grid != 0) {  // panels are shared
        const bool ragged = units % p.grid != 0 || (per % p.slabs != 0 && p.slabs % per != 0);
        const long sharers = div_up(p.slabs, per) + (ragged ? 1 : 0);
        t += c.exchange + c.share * (float)(sharers < p.slabs ? sharers : p.slabs) * 16 * p.wn * padded * 4 / 1024.f;
    }
    return t;
}

// 17 to 64 rows that the skinny GEMM's planner gives to its workgroup kernel.  That kernel was tuned on weights whose rows and k deal out in whole
// panels and slabs over the compute units; elsewhere the shares of a panel lie with up to twenty workgroups, whose sums one of them collects.  Over 1079
// such calls (n and k drawn from 1024 to 28672, 40 % of them multiples of 256, 512 or 1024; row-major and packed) the choice below is 17 % faster in
// the mean with weights from memory and 25 % with weights from the 256 MB cache: 57 x 2832 x 1792 13.3 -> 6.4 us / 14.5 -> 6.4, 50 x 6176 x 3072 15.4 -> 11.2 / 15.5 ->
// 8.5, 57 x 1752 x 14592 19.5 -> 12.0 from the cache, 64 x 11096 x 5120 21.8 -> 20.1 / 21.5 -> 13.7.  The margins are for the fits' errors: whole panels, where
// nothing is exchanged, and weights above 76 MB, where memory bounds both, are predicted less well.  Twelve of the 1079 lose more than 3 % from one of the two, one more
// than 8 % (57 x 8192 x 8192 from memory 10 %, and from the cache 10 % faster).  Above 112 MB all stay, though not for want of gains: on their best tile plan
// the 114 sizes there are 6 % slower in the mean from memory and 21 % faster from the cache (49 x 14744 x 9216 26 and 51 % faster, 19 x 16616 x 13824 33 and 22 % slower;
// 64 x 8192 x 28672 44 us, 50 on tiles), and the fits do not tell them apart.
// Three kinds of sizes outside that range stay: k up to 1024 with more tiles than two rounds of compute units (37 x 45056 x 768 13.0 / 14.6 us, weight from the
// cache; of 260 drawn n from 32776 to 128056 the costs put 16 on tiles, the six of them with k = 768 4 % slower in the mean there, the ten from k = 1280 on 6 % faster), k of
// one chunk, and, up to 32 rows, k of one or two slabs (34 x 45008 x 256 packed 6.6 / 11.0, 32 x 42896 x 256 packed 5.5 / 11.0, 22 x 16792 x 512 packed 5.8 / 7.0, 30 x
// 608 x 1024 packed 4.9 / 5.5), unless the panels take a second round and the tiles do not (22 x 10352 x 1024 6.7 / 5.8) or k is two slabs (16390 to 32768 columns of k = 1024,
// which then go by the costs: 69 drawn ones 13 % faster from the cache and 4 % from memory).
// The row-split and K-split kernels stay: the tiled kernel is 3 to 60 % slower than they are on all but a few of their sizes.
bool tiled_instead(int m, int n, int k, const hfrk_gemm_plan& skinny, hfrk_tiled_plan* plan) {
    if (m <= 16 || skinny.wn < 1 || (long)n * k > (112L << 20) || !tiled_size_ok(m, n, k)) return false;
    if (k <= (n > 64 * 2 * kNumCU ? 1024 : 256)) return false;
    if (m <= 32 && skinny.slabs < 3 && (skinny.panels <= skinny.grid || (skinny.slabs == 1 && div_up(n, 64) > kNumCU))) return false;
    const bool whole_panels = skinny.panels % skinny.grid == 0, large = (long)n * k > (76L << 20);
    const float margin = (whole_panels ? 1.08f : 1.03f) + (large ? .05f : 0.f);
    return margin * make_few_rows_plan(m, n, k, kTiledMaxSplits, plan) < workgroup_kernel_cost(m, n, k, skinny);
}

static void make_tiled_plan(int m, int n, int k, int max_splits, hfrk_tiled_plan* plan) {
    float best = INFINITY;
    const int stages = div_up(k, kTiledStage);
    if (m <= 64) {  // (the fit below starts at 65 rows)
        make_few_rows_plan(m, n, k, max_splits, plan);
        return;
    }
    for (int shape = 0; shape < kTiledShapeCount; ++shape) {
        const TiledShape& s = kTiledShapes[shape];
        const int tiles_m = div_up(m, s.bm);
        const long tiles = (long)tiles_m * div_up(n, s.bn);
        for (int splits = 1; splits <= max_splits && splits <= stages; ++splits) {
            // a split keeps at least two stages, the launch at most two workgroups per compute unit, and the partial tiles fit the
            // stream's workspace (256 x 256 tiles: 256 of them)
            if (splits > 1 && (tiles * splits > 2 * kNumCU || stages < 2 * splits || tiled_ws_bytes(s, m, n, splits) > kWsFloats * sizeof(float))) break;
            const float t = tiled_cost(m, n, k, shape, splits);
            if (t < best) {
                best = t;
                plan->shape = shape;
                plan->splits = splits;
                // the 32 workgroups of an XCD cover about as many rows as columns of D
                const int square = (int)lroundf(sqrtf(32.f * s.bn / s.bm));
                plan->group_m = tiles_m < square ? tiles_m : square;
            }
        }
    }
}

// The workgroups of an XCD share rows of A and of the weight.  Walking k in step they all ask for a line while it is on its way into their
// L2, and where rows are a multiple of some KB apart they all ask the same channels.  So each starts at a stage of its own: row and column of
// tiles turn the start so that those who share an operand are spread evenly, within a window of k whose operands (of the workgroups that an XCD
// runs at a time) take 700 KB of its 4 MB L2; a window of one stage is no turn.  As layer calls with the quantisation in front, us: 201 x 6144 x
// 4096 16.1 -> 15.3, 300 x 4096 x 4096 16.9 -> 15.9, 512 x 4096 x 14336 packed 40.9 -> 39.2, 474 x 11744 x 11520 packed 78.3 -> 72.6, 507 x 14160 x
// 15872 115 -> 109, 3385 x 2352 x 25600 packed 328 -> 289, 3605 x 2392 x 18928 242 -> 210; the worst 209 x 6752 x 3328 14.8 -> 15.0, 156 x 7920 x 2848
// 16.0 -> 16.3.  Windows of 400 KB gain a third of that, of 1.2 to 3 MB as much on the sizes above and lose up to 7 % on others (1192 x 5488 x 2048 23.1 ->
// 24.6); k turned as a whole loses up to twice the time where it does not fit L2.  64 x 64 tiles start together: they lose 1 to 3 % by it
// (187 x 4024 x 7872 21.6 -> 22.2, 317 x 1800 x 6400 18.2 -> 18.7).
static void turn_k(TiledGemmArgs* a, int shape) {
    const TiledShape& s = kTiledShapes[shape];
    const int grid = a->tiles_m * a->tiles_n * a->splits, resident = kNumCU * s.per_cu;
    const int per_xcd = div_up(grid < resident ? grid : resident, 8);
    int columns = div_up(per_xcd, a->group_m);
    columns = columns < a->tiles_n ? columns : a->tiles_n;
    a->phase_m = 65536 / a->group_m;
    a->phase_n = 65536 / columns;
    a->window = shape == 4 ? 1 : (int)(700 * 1024 / (((long)a->group_m * s.bm + (long)columns * s.bn) * kTiledStage));
    a->window = a->window < 1 ? 1 : a->window;
}

int tiled_launch(const void* A, const void* B, bool packed, void* D, const void* base, int base_stride, const float* scale_a, int sa_stride,
                 const float* scale_b, int sb_stride, int m, int n, int k, int b_stride, int d_dtype, const hfrk_tiled_plan& p, float* ws, size_t ws_bytes,
                 int* counters, hipStream_t stream) {
    const TiledShape& s = kTiledShapes[p.shape];
    const int row_tiles = div_up(m, s.bm);
    if ((uint64_t)row_tiles * div_up(n, s.bn) * p.splits * s.threads >> 32) {
        // A launch holds fewer than 2^32 threads: 2^23 tiles or more that a plan cuts 64 columns wide go as two launches (or, halved once more,
        // up to four), each of half the rows of tiles.  k is not split then, as the partial sums of so many tiles fit no workspace.
        const int half = row_tiles / 2, rows = half * s.bm;
        auto part = [&](int row, int count) {
            const hfrk_tiled_plan q{p.shape, p.splits, p.group_m < half ? p.group_m : half};
            return tiled_launch(static_cast<const uint8_t*>(A) + (size_t)row * k, B, packed, static_cast<uint8_t*>(D) + (size_t)row * n * 2,
                                base ? static_cast<const uint8_t*>(base) + (size_t)row * base_stride * 2 : base, base_stride, scale_a + (size_t)row * sa_stride,
                                sa_stride, scale_b, sb_stride, count, n, k, b_stride, d_dtype, q, ws, ws_bytes, counters, stream);
        };
        const int rc = part(0, rows);
        return rc == HFRK_SUCCESS ? part(rows, m - rows) : rc;
    }
    TiledGemmArgs args{};
    args.A = static_cast<const uint8_t*>(A);
    args.B = static_cast<const uint8_t*>(B);
    args.D = D;
    args.base = base;
    args.base_stride = base ? base_stride : 0;
    args.scale_a = scale_a;
    args.scale_b = scale_b;
    args.sa_stride = sa_stride;
    args.sb_stride = sb_stride;
    args.m = m;
    args.n = n;
    args.k = k;
    args.b_stride = b_stride;
    args.d_dtype = d_dtype;
    args.vec = n % 8 == 0 && args.base_stride % 8 == 0 && ((reinterpret_cast<uintptr_t>(D) | reinterpret_cast<uintptr_t>(base)) & 15) == 0;
    args.tiles_m = row_tiles;
    args.tiles_n = div_up(n, s.bn);
    args.group_m = p.group_m;
    const int stages = div_up(k, kTiledStage);
    args.splits = p.splits;
    args.ws = ws;
    args.ws_bytes = (uint32_t)ws_bytes;
    args.counters = counters;
    args.stages_q = stages / p.splits;
    args.stages_r = stages % p.splits;
    turn_k(&args, p.shape);
    return packed ? launch_tiled_packed(args, p.shape, stream)
                  : launch_tiled_rowmajor(args, p.shape, stream);
}

}  // namespace hfrk

extern "C" {

int hfrk_tiled_gemm_plan(int m, int n, int k, hfrk_tiled_plan* plan) {
    if (!plan || !hfrk::tiled_size_ok(m, n, k)) return HFRK_BAD_SHAPE;
    if (k % 16 != 0) return HFRK_K_NOT_DIVISIBLE_BY_WARPTILE_K;
    hfrk::make_tiled_plan(m, n, k, hfrk::kTiledMaxSplits, plan);
    return HFRK_SUCCESS;
}

int hfrk_tiled_gemm(const void* A, const void* B, int packed, void* D, const void* base, int base_stride, const float* scale_a,
                    int sa_stride, const float* scale_b, int sb_stride, int m, int n, int k, int b_stride, int d_dtype,
                    const hfrk_tiled_plan* plan, void* stream) {
    using namespace hfrk;
    if (packed) b_stride = k;
    if (!tiled_size_ok(m, n, k) || b_stride < k || b_stride > (1 << 21)) return HFRK_BAD_SHAPE;
    if (k % 16 != 0 || (packed && k % 256 != 0)) return HFRK_K_NOT_DIVISIBLE_BY_WARPTILE_K;
    if (d_dtype != HFRK_F16 && d_dtype != HFRK_BF16) return HFRK_BAD_DTYPE;
    if (!A || !B || !D || !scale_a) return HFRK_BAD_SHAPE;
    if ((sa_stride != 0 && sa_stride != 1) || (sb_stride != 0 && sb_stride != 1)) return HFRK_BAD_SHAPE;
    if (base && base_stride != 0 && (base_stride < n || base_stride > (1 << 21))) return HFRK_BAD_SHAPE;
    if ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B)) & 15 || (b_stride & 15)) return HFRK_BAD_ALIGNMENT;
    if ((reinterpret_cast<uintptr_t>(D) | reinterpret_cast<uintptr_t>(base)) & 1) return HFRK_BAD_ALIGNMENT;
    hfrk_tiled_plan p;
    if (plan) {
        p = *plan;
        const int rc = check_tiled_plan(m, n, k, p);
        if (rc != HFRK_SUCCESS) return rc;
    } else {
        make_tiled_plan(m, n, k, kTiledMaxSplits, &p);
    }
    float* ws = nullptr;
    size_t ws_bytes = 0;
    int* counters = nullptr;
    if (p.splits > 1) {
        const int rc = stream_workspace(static_cast<hipStream_t>(stream), &ws, &ws_bytes, &counters);
        if (rc != HFRK_SUCCESS) {
            // no workspace left, no memory for one (a caching allocator may hold it all), or none before a capture began: a call that names
            // no plan runs without splitting k
            const bool none = rc == HFRK_NO_WORKSPACE || rc == HFRK_NOT_INITIALISED || (rc == HFRK_HIP_ERROR && hfrk_last_hip_error() == (int)hipErrorOutOfMemory);
            if (plan || !none) return rc;
            make_tiled_plan(m, n, k, 1, &p);
        }
    }
    return tiled_launch(A, B, packed != 0, D, base, base_stride, scale_a, sa_stride, scale_b, sb_stride, m, n, k, b_stride, d_dtype, p, ws, ws_bytes,
                        counters, static_cast<hipStream_t>(stream));
}

}  // extern "C"
