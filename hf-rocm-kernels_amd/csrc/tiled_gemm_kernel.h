// Tiled FP8 (OCP e4m3fn) GEMM for more rows than the skinny kernels take:
//   D[m,n] = (base ? base[m,n] : 0) + sa[m] * sb[n] * sum_k A[m,k] * W[n,k]
// No counterpart in the reference, whose kernel stops at 32 rows (skinny_gemm_caller.cu:33-60); the linear layer ran such calls
// as one skinny launch per 64 rows, each of which streamed the whole weight again.
//
//  * A wave owns TM x TN matrix tiles of 32 x 32 (v_mfma_f32_32x32x64_f8f6f4, 64 cycles each).  The largest tile (256 x 256) runs on eight
//    waves of 128 x 64, two per SIMD: with four of 128 x 128 an operand byte read from LDS fed a third more multiply-adds, but nothing ran
//    while the one wave of a SIMD waited for its stage or stored (4096 x 28672 x 4096 432 -> 409 us, 4096 x 4096 x 4096 62.7 -> 57,
//    2048 x 6144 x 4096 56 -> 52; 12 % in the mean over 70 weights and rows where tiles are few).  The 256 x 128 tile has eight
//    waves of 64 x 64 for the same reason (four of 128 x 64 before: 4096 x 6144 x 4096 106 -> 97 us, 4096 x 2048 x 2048 23.0 -> 21.0,
//    300 x 20000 x 4096 56.3 -> 53.5, 1024 x 8192 x 8192 64.6 -> 64; 512 x 10240 x 8192 54.6 -> 55.4 is the loss), but for a long k in rows that
//    begin inside a 128-byte line, where four are the faster (tiled_gemm_rowmajor.hip).  A long k on the largest tile is what eight cost
//    there: 2513 x 11824 x 13312 314 -> 322, 1415 x 6304 x 18944 188 -> 193.  The others have four waves, one per SIMD: 128 x 128 on
//    eight or sixteen takes the same time.
//  * Bound (counters in profiles/tiled_gemm_counters_and_plans.txt, shares of the cycles in which a compute unit has work): 4096 x 28672 x
//    4096 matrix cores 68 %, at the clock their power leaves, LDS 30 % (62 and 19 on four waves); 512 x 4096 x 14336 packed 52 and 40 %;
//    201 x 6144 x 4096 32 and 27 %.
//    The small tiles wait for what a compute unit fetches, 135 GB/s from its L2 and 58 where a stage waits for lines from memory: loads
//    alone, without matrix instructions and operand reads, take 7 us of 201 x 6144 x 4096 with everything in L2, 10 from the 256 MB cache and
//    15.6 from memory, with three stages in flight or six.
//  * On every tile but the largest four more waves do nothing but load, one per SIMD.  A compute unit takes a load instruction of 1 KB in 16
//    cycles and holds back the wave whose turn has not come: where the multiplying waves loaded for themselves, a stage took about as long as its
//    loads and its matrix instructions after one another (201 x 6144 x 4096 with the weight in the 256 MB cache: 11.6 us without matrix instructions
//    and operand reads, 9.0 without loads, 15.4 whole).  Now, weight in that cache / from memory: that size 14.1 -> 13.0 / 17.0 -> 17.0, 512 x
//    4096 x 4096 18.1 -> 15.8 / 22.1 -> 22.1, 65 x 4096 x 4096 10.7 -> 9.1 / 11.2 -> 10.6, 244 x 2752 x 3072 9.3 -> 8.2 / 10.2 -> 9.8, 1024 x 4096 x
//    4096 25.5 -> 23.3 / 29.1 -> 28.9; the worst 64 x 8192 x 28672 49.2 -> 50.1 / 50.1 -> 50.3 and, packed, 84 x 8088 x 3584 9.9 -> 9.4 / 11.0 ->
//    11.5.  Eight loading waves are no faster, a higher priority for either kind changes nothing.  The tiles whose waves hold 128 x 64 (TM = 4)
//    have no registers left for a third wave per SIMD.
//  * Operands go from memory to LDS without passing registers (buffer_load_dwordx4 ... lds), NST stages of 128 bytes of k deep, the
//    stage NST ahead being requested behind the barrier that frees its slot.  One barrier per stage: a wave reads the operands of
//    k step s + 1 (64 bytes) while it multiplies those of step s, so nothing in a step waits for LDS but its first instruction.
//  * The 256 x 256 tile has room for two such stages, which left a load one stage to arrive in, so LDS holds five halves instead (64 bytes of
//    k each): a stage is requested when the first half of the one before it is free, one and a half stages ahead.  A load then covers 64 bytes
//    of 16 rows, the two halves of a line one after the other.  Two stages -> five halves, weight in the 256 MB cache / from memory: 4096 x
//    28672 x 4096 396 -> 384 / 398 -> 384 us, 2048 x 28672 x 4096 219 -> 212 / 221 -> 213, 418 x 16920 x 6656 packed 74.1 -> 68.4 / 75.4 -> 68.7,
//    1024 x 8192 x 8192 in 2 splits 75.8 -> 72.2 / 75.7 -> 72.9, 4096 x 4096 x 4096 58.4 -> 57.3 / 58.7 -> 57.9.  On operands of zeros the first takes
//    313 us and took 345: the rest of it is the clock that the matrix cores' power leaves.
//  * Such a load fills LDS in lane order, so the swizzle that keeps operand reads free of bank conflicts is applied to the memory
//    side: the lane that fills slot c of row r fetches piece c ^ f(r) of that row (a permutation within one 128-byte line).
//    Measured conflicts: 3.5 % of the LDS cycles on the 256 x 256 tile, 1 - 2 % on the smaller ones.  A packed weight is fetched as
//    512-byte runs into the same kind of layout; its operand reads do conflict (128 x 128: a third of the LDS cycles).
//  * Rows and columns past the edge, and the part of the last stage past k, are outside the buffers' ranges and read as zero.
//  * Weights are the matrix instruction's A operand with their rows permuted so that a lane's 16 results of a tile are consecutive
//    columns; results go through LDS in fp32 and leave as whole rows, scaled, added to their addend and rounded once.
//  * Workgroup ids are dealt to the XCDs in contiguous ranges and walk the tiles in column-major groups of group_m rows of tiles, so
//    that the workgroups of one L2 share both operands.
//  * Few tiles and a long k: k is cut between `splits` workgroups.  Partial tiles are written through to memory, the last arriver
//    adds them in split order (bit-reproducible), its own from its registers.
//
// Measured (us, bf16 out): 4096 x 28672 x 4096 384 - 398 (2.42 - 2.51 PFLOP/s; 1550 as 64 skinny launches; a loop that stays resident clocks at 1.8 - 2.0
// GHz, so the matrix cores' power bounds it before their issue rate does), 512 x 4096 x 14336 packed 33 (150), 201 x 6144 x 4096
// 12 (46), 65 x 4096 x 4096 9.1 (16).  The epilogue is written with little code on
// purpose: with a branch per value for NaN and 64-bit addresses it took 18 us of a 256 x 256 tile, now 7.
#pragma once

#include "tiled_gemm.h"

namespace hfrk {

typedef float v16f __attribute__((ext_vector_type(16)));

// One 16-byte-per-lane load from memory straight into LDS: lane l's piece lands at lds_base + 16 l.  As inline assembly because the
// compiler, when it knows of such a load, waits for it before every LDS read that follows; the waits are placed by hand here.  m0 is
// reserved: the compiler sets it in front of each use of its own, and a clobber list may not name it.
__device__ __forceinline__ void load_to_lds(const v4i& rsrc, int voffset, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds_base), "v"(voffset), "s"(rsrc) : "memory");
}

// All but the COUNT youngest loads of this wave have landed, and its LDS reads are done.
template <int COUNT>
__device__ __forceinline__ void wait_loads_and_lds() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(COUNT) : "memory");
}

__device__ __forceinline__ void workgroup_barrier() { asm volatile("s_barrier" ::: "memory"); }

__device__ __forceinline__ v4i tile_rsrc(const uint8_t* base, uint32_t bytes) {
    const uint64_t p = reinterpret_cast<uint64_t>(base);
    return v4i{__builtin_amdgcn_readfirstlane((int)(uint32_t)p), __builtin_amdgcn_readfirstlane((int)((uint32_t)(p >> 32) & 0xffffu)),
               __builtin_amdgcn_readfirstlane((int)bytes), 0x00020000};
}

// Two floats to two 16-bit values in one register, round to nearest even (v_cvt_pk_bf16_f32 / v_cvt_pk_f16_f32: no branch for NaN).
template <int DT>
__device__ __forceinline__ uint32_t pack_pair(float lo, float hi) {
    typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
    typedef _Float16 v2h __attribute__((ext_vector_type(2)));
    if constexpr (DT == HFRK_BF16) return __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{lo, hi}, v2bf));
    else return __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{lo, hi}, v2h));
}

// LW: waves that only load.
template <int TM, int TN, int WM, int WN, int NST, int WGS, bool PACKED, int LW>
__global__ void __launch_bounds__(64 * (WM * WN + LW), WGS * (WM * WN + LW) / 4) tiled_gemm_kernel(const TiledGemmArgs a) {
    constexpr int NW = WM * WN, NL = LW ? LW : NW;  // waves that multiply, that load
    constexpr int BM = 32 * TM * WM, BN = 32 * TN * WN;
    constexpr int KB = kTiledStage;
    constexpr int A_BYTES = BM * KB, B_BYTES = BN * KB, STAGE = A_BYTES + B_BYTES;
    constexpr int LA = A_BYTES / (1024 * NL), LB = B_BYTES / (1024 * NL);  // load instructions per loading wave and stage, 1 KB each
    constexpr int NMMA = TM * TN;
    // NST counts whole stages, or (HALF) the halves of stages, 64 bytes of k each, that LDS holds.
    constexpr bool HALF = tiled_half_stages(TM, NW);
    constexpr int ROW = HALF ? KB / 2 : KB, SLOT = HALF ? STAGE / 2 : STAGE, RING = NST * SLOT, AHEAD = HALF ? NST / 2 : NST;  // AHEAD: stages requested in front
    constexpr int kOutside = 0x7ffffff0;  // beyond any tile's range

    extern __shared__ __align__(16) uint8_t lds[];
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((int)(uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void*)lds));

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int loader = wave - (LW ? NW : 0);  // number among the waves that load
    const int wm = wave / WN, wn = wave % WN;
    const int lr = lane & 31, lg = lane >> 5;

    // ---- which tile, which part of k ---------------------------------------------------------------------------------
    int id = blockIdx.x;
    {
        const int per = (int)gridDim.x >> 3, extra = (int)gridDim.x & 7, x = id & 7;  // XCD x works on one contiguous range of ids
        id = x * per + min(x, extra) + (id >> 3);
    }
    const int tiles = a.tiles_m * a.tiles_n;
    const int split = a.splits == 1 ? 0 : id / tiles, tile = id - split * tiles;  // neighbours work on the same part of k
    const int group_tiles = a.group_m * a.tiles_n;
    const int grp = tile / group_tiles, in_grp = tile - grp * group_tiles;
    const int gm = min(a.group_m, a.tiles_m - grp * a.group_m);
    const int tn = in_grp / gm, tm = grp * a.group_m + in_grp - tn * gm;
    const int m0 = tm * BM, n0 = tn * BN;
    const uint32_t phase = ((uint32_t)(in_grp - tn * gm) * (uint32_t)a.phase_m + (uint32_t)tn * (uint32_t)a.phase_n) & 0xffff;  // in 65536ths
    const int s_begin = split * a.stages_q + min(split, a.stages_r), s_end = s_begin + a.stages_q + (split < a.stages_r ? 1 : 0);

    // ---- operand streams ---------------------------------------------------------------------------------------------
    // buffers over this tile's rows, moved to the stage that is requested
    const int rows_a = min(BM, a.m - m0);
    v4i ra = tile_rsrc(a.A + (long)m0 * a.k, (uint32_t)rows_a * (uint32_t)a.k);
    v4i rb;
    constexpr int kStepB = PACKED ? 2048 : KB;  // a stage of a packed 16-row tile is half of a 4 KB chunk
    if constexpr (PACKED) {
        const int tiles16 = min(BN / 16, (a.n + 15) / 16 - n0 / 16);
        rb = tile_rsrc(a.B + (long)(n0 / 16) * a.k * 16, (uint32_t)tiles16 * (uint32_t)a.k * 16u);
    } else {
        const int rows_b = min(BN, a.n - n0);
        rb = tile_rsrc(a.B + (long)n0 * a.b_stride, (uint32_t)(rows_b - 1) * (uint32_t)a.b_stride + (uint32_t)a.k);
    }
    int va[LA], vb[LB];
    int pa[LA], pb[LB];  // k byte of the lane's piece within its stage (for the last, partial stage)
#pragma unroll
    for (int q = 0; q < LA; ++q) {
        const int row = HALF ? ((q >> 1) * NL + loader) * 16 + (lane >> 2) : (q * NL + loader) * 8 + (lane >> 3);
        pa[q] = HALF ? ((lane & 3) ^ ((row >> 2) & 3)) * 16 + (q & 1) * ROW : ((lane & 7) ^ ((row >> 1) & 7)) * 16;
        va[q] = row * a.k + pa[q];
    }
#pragma unroll
    for (int q = 0; q < LB; ++q) {
        if constexpr (PACKED) {
            // LDS block (16-row tile, half of the stage): [piece j][k group][row slot], 1 KB
            const int blk = HALF ? ((q >> 1) * NL + loader) * 2 + (q & 1) : q * NL + loader, t16 = blk >> 1, s = blk & 1, group = (lane >> 4) & 1;
            const int row = (lane & 15) ^ ((t16 & 1) << 3) ^ group << 2;
            vb[q] = t16 * a.k * 16 + (lane >> 5) * 1024 + s * 512 + group * 256 + row * 16;
            pb[q] = 0;
        } else {
            const int row = HALF ? ((q >> 1) * NL + loader) * 16 + (lane >> 2) : (q * NL + loader) * 8 + (lane >> 3);
            pb[q] = HALF ? ((lane & 3) ^ (((row >> 2) & 1) | ((row >> 4) & 1) << 1)) * 16 + (q & 1) * ROW
                         : ((lane & 7) ^ (((row >> 1) & 3) | ((row >> 4) & 1) << 2)) * 16;
            vb[q] = row * a.b_stride + pb[q];
        }
    }
    // The stages of a window of k are requested from `phase` of it on and round to there; then those of the next window.
    int issued = s_begin, window = s_begin, window_end = min(s_begin + a.window, s_end), window_left = window_end - window;
    int at = window + (int)((phase * (uint32_t)window_left) >> 16);  // the stage to request next
    const uint64_t base_a = (uint64_t)(uint32_t)ra[1] << 32 | (uint32_t)ra[0], base_b = (uint64_t)(uint32_t)rb[1] << 32 | (uint32_t)rb[0];
    const int range_a = ra[2], range_b = rb[2];
    uint32_t slot_issue = 0, slot_issue_odd = SLOT;  // where the next stage goes (HALF: its first and second half)
    auto next_slot = [](uint32_t slot) __attribute__((always_inline)) { return slot + SLOT == RING ? 0u : slot + SLOT; };
    const int k_tail = a.k & (KB - 1), tail_stage = k_tail ? a.k / KB : -1;
    auto issue_begin = [&]() __attribute__((always_inline)) {
        auto seek = [&](v4i& r, uint64_t base, int range, int by) __attribute__((always_inline)) {
            const uint64_t p = base + (uint32_t)by;
            r[0] = (int)(uint32_t)p;
            r[1] = (int)(uint32_t)(p >> 32);
            r[2] = issued < s_end ? range - by : 0;  // past the end: as many loads as ever, nothing is read
        };
        seek(ra, base_a, range_a, at * KB);
        seek(rb, base_b, range_b, at * kStepB);
    };
    auto issue_a = [&](int q) __attribute__((always_inline)) {
        int off = va[q];
        if (at == tail_stage) off = pa[q] < k_tail ? off : kOutside;
        load_to_lds(ra, off, lds0 + (HALF && (q & 1) ? slot_issue_odd : slot_issue) + (uint32_t)((HALF ? q >> 1 : q) * NL + loader) * 1024u);
    };
    auto issue_b = [&](int q) __attribute__((always_inline)) {
        int off = vb[q];
        if (!PACKED && at == tail_stage) off = pb[q] < k_tail ? off : kOutside;
        load_to_lds(rb, off, lds0 + (HALF && (q & 1) ? slot_issue_odd : slot_issue) + ROW * BM + (uint32_t)((HALF ? q >> 1 : q) * NL + loader) * 1024u);
    };
    auto issue_end = [&]() __attribute__((always_inline)) {
        ++issued;
        at = at + 1 == window_end ? window : at + 1;
        if (--window_left == 0) {
            window = window_end;
            window_end = min(window_end + a.window, s_end);
            window_left = window_end - window;
            at = window + (int)((phase * (uint32_t)window_left) >> 16);
        }
        slot_issue = next_slot(HALF ? slot_issue_odd : slot_issue);
        slot_issue_odd = next_slot(slot_issue);
    };

    // ---- operand reads -----------------------------------------------------------------------------------------------
    // matrix row r of a weight tile is weight row perm(r): a lane's 16 results of a tile are then 16 consecutive columns
    const int perm = ((lr >> 2) & 1) * 16 + (lr >> 3) * 4 + (lr & 3);
    const int fa = HALF ? (lr >> 2) & 3 : (lr >> 1) & 7, fb = HALF ? ((perm >> 2) & 1) | ((perm >> 4) & 1) << 1 : ((perm >> 1) & 3) | ((perm >> 4) & 1) << 2;
    const int a_row = (wm * TM * 32 + lr) * ROW;
    const int b_row = ROW * BM + (PACKED ? (wn * TN * 2 + (perm >> 4)) * 16 * ROW + lg * 256 + ((perm & 15) ^ ((perm >> 4) << 3) ^ (lg << 2)) * 16
                                        : (wn * TN * 32 + perm) * ROW);
    uint32_t slot_read = 0;
    v8i fra[2][TM], frb[2][TN];
    auto read16 = [&](int off) __attribute__((always_inline)) { return *reinterpret_cast<const v4i*>(lds + off); };
    auto join = [](v4i lo, v4i hi) __attribute__((always_inline)) { return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}; };
    auto read_a = [&](v8i& dst, int i, int s) __attribute__((always_inline)) {
        const int off = (int)slot_read + a_row + (((2 * lg) ^ fa ^ (HALF ? 0 : 4 * s)) << 4);
        dst = join(read16(off + i * 32 * ROW), read16((off ^ 16) + i * 32 * ROW));
    };
    auto read_b = [&](v8i& dst, int j, int s) __attribute__((always_inline)) {
        if constexpr (PACKED) {
            const int off = (int)slot_read + b_row + j * 32 * ROW + (HALF ? 0 : s * 1024);
            dst = join(read16(off), read16(off + 512));
        } else {
            const int off = (int)slot_read + b_row + (((2 * lg) ^ fb ^ (HALF ? 0 : 4 * s)) << 4);
            dst = join(read16(off + j * 32 * ROW), read16((off ^ 16) + j * 32 * ROW));
        }
    };

    v16f acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

    // Half a stage (64 bytes of k): multiply the operands read half a stage ago (register set S) while the next half's are read into
    // the other set.  The second half reads from the next stage, so it opens with the wait for that stage and a barrier behind it.  With
    // whole stages in LDS that barrier also frees this stage's slot, and the stage NST ahead is requested into it behind the barrier.
    // With halves, the first half's slot is free half a stage earlier, behind a barrier of its own: the five halves then hold one that is
    // being read, a whole stage in flight, and the two into which the stage after that is requested.
    // The schedule is fixed: operand reads in front of the first three quarters of the matrix instructions, loads spread over all of them.
    constexpr int kFirstLoads = HALF ? (LA + LB) / 2 : 0;  // of a stage's loads, those in the first half
    auto half = [&](auto sel) __attribute__((always_inline)) {
        constexpr int S = decltype(sel)::value;
        if constexpr (HALF && S == 0) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            workgroup_barrier();
            issue_begin();
        }
        if constexpr (S == 1) {
            if constexpr (HALF) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kFirstLoads) : "memory");
            else if constexpr (LW) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            else wait_loads_and_lds<(NST - 2) * (LA + LB)>();
            workgroup_barrier();
            if constexpr (!LW && !HALF) issue_begin();
        }
        if constexpr (HALF || S == 1) slot_read = next_slot(slot_read);
        constexpr int READS = TM + TN, FIRST = S == 1 ? kFirstLoads : 0;
        constexpr int LOADS = LW ? 0 : HALF ? (S == 0 ? kFirstLoads : LA + LB - kFirstLoads) : S == 1 ? LA + LB : 0;
        int reads = 0, loads = 0;
#pragma unroll
        for (int t = 0; t < NMMA; ++t) {
            const int reads_to = NMMA <= 2 ? READS : min(READS, (t + 1) * READS * 4 / (3 * NMMA) + 1), loads_to = min(LOADS, (t + 1) * LOADS / NMMA);
#pragma unroll
            for (int r = 0; r < READS; ++r)
                if (r >= reads && r < reads_to) {
                    if (r < TN) read_b(frb[S ^ 1][r], r, S ^ 1);
                    else read_a(fra[S ^ 1][r - TN], r - TN, S ^ 1);
                }
#pragma unroll
            for (int l = 0; l < LOADS; ++l)
                if (l >= loads && l < loads_to) {
                    if (FIRST + l < LA) issue_a(FIRST + l);
                    else issue_b(FIRST + l - LA);
                }
            reads = reads_to;
            loads = loads_to;
            acc[t / TN][t % TN] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(frb[S][t % TN], fra[S][t / TN], acc[t / TN][t % TN], 0, 0, 0, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (S == 1 && !LW) issue_end();
    };

    // ---- main loop ---------------------------------------------------------------------------------------------------
    auto issue_stage = [&]() __attribute__((always_inline)) {
        issue_begin();
#pragma unroll
        for (int q = 0; q < LA; ++q) issue_a(q);
#pragma unroll
        for (int q = 0; q < LB; ++q) issue_b(q);
        issue_end();
    };
    if (!LW || wave >= NW) {
        // A load may read a scalar that a vector instruction wrote (v_readfirstlane) only five cycles later, and nobody looks after that
        // for a load in inline assembly: both buffers pass through the wait.  From here on scalar instructions move them.
        asm volatile("s_nop 4" : "+s"(ra), "+s"(rb) : : "memory");
#pragma unroll 1
        for (int s = 0; s < AHEAD; ++s) issue_stage();
        wait_loads_and_lds<(AHEAD - 1) * (LA + LB)>();
        if constexpr (LW) {  // the barriers of the multiplying waves: one in front of the loop, one per stage, one behind the loop
            workgroup_barrier();
#pragma unroll 1
            for (int s = s_begin; s < s_end; ++s) {
                wait_loads_and_lds<(NST - 2) * (LA + LB)>();
                workgroup_barrier();
                issue_stage();
            }
            wait_loads_and_lds<0>();
            workgroup_barrier();
            return;  // later barriers wait for the waves that are left
        }
    }
    workgroup_barrier();
#pragma unroll
    for (int j = 0; j < TN; ++j) read_b(frb[0][j], j, 0);
#pragma unroll
    for (int i = 0; i < TM; ++i) read_a(fra[0][i], i, 0);
#pragma unroll 1
    for (int s = s_begin; s < s_end; ++s) {
        half(std::integral_constant<int, 0>{});
        half(std::integral_constant<int, 1>{});
    }
    wait_loads_and_lds<0>();
    workgroup_barrier();  // LDS is free: no wave reads operands any more, no load is under way

    // ---- partial sums of a tile whose k is split -----------------------------------------------------------------------
    if (a.splits > 1) {
        const __amdgpu_buffer_rsrc_t ws = make_rsrc(a.ws, a.ws_bytes);
        constexpr int kCoherent = 17;  // sc0 | sc1: written through to memory, read past the caches (the XCDs' L2s are not coherent)
        auto ws_off = [&](int sp, int t, int p) __attribute__((always_inline)) {
            return ((((tile * a.splits + sp) * NW + wave) * NMMA + t) * 4 + p) * 1024 + lane * 16;
        };
#pragma unroll
        for (int t = 0; t < NMMA; ++t)
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const v16f& x = acc[t / TN][t % TN];
                const v4f v = {x[4 * p], x[4 * p + 1], x[4 * p + 2], x[4 * p + 3]};
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4i, v), ws, ws_off(split, t, p), 0, kCoherent);
            }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        int* const flag = reinterpret_cast<int*>(lds);
        if (tid == 0) {
            const int seen = __hip_atomic_fetch_add(a.counters + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const int last = seen == a.splits - 1;
            if (last) __hip_atomic_store(a.counters + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *flag = last;
        }
        __syncthreads();
        const int last = *flag;
        __syncthreads();  // the epilogue writes where the flag lies
        if (!last) return;
        // The last arriver adds the partials in split order, its own from its registers; the others' are requested FLY at a time.  What it costs
        // is the round trips: with its own read back and one split at a time 512 x 4096 x 14336 in 2 splits 43.8 -> 43.0 us, 64 x 4096 x 14336 in
        // 4 17.5 -> 17.1, 1024 x 8192 x 8192 on 256 x 256 tiles in 2 82 -> 76.
        // CH matrix tiles' shares of FLY splits are in flight together: what fits the registers.
        constexpr int CH = NMMA == 1 || WGS * (NW + LW) > 8 || (LW == 0 && NW > 4) ? 1 : 2, FLY = NMMA == 1 ? 7 : 3;
#pragma unroll
        for (int t0 = 0; t0 < NMMA; t0 += CH) {
            v4f sum[CH * 4];
#pragma unroll
            for (int p = 0; p < CH * 4; ++p) sum[p] = v4f{0.f, 0.f, 0.f, 0.f};
            auto add_shares = [&](int first, int end) __attribute__((always_inline)) {
#pragma unroll 1
                for (; first < end; first += FLY) {
                    v4i share[FLY][CH * 4];
#pragma unroll
                    for (int j = 0; j < FLY; ++j)
                        if (first + j < end) {
#pragma unroll
                            for (int p = 0; p < CH * 4; ++p)
                                share[j][p] = __builtin_amdgcn_raw_buffer_load_b128(ws, ws_off(first + j, t0 + p / 4, p % 4), 0, kCoherent);
                        }
#pragma unroll
                    for (int j = 0; j < FLY; ++j)
                        if (first + j < end) {
#pragma unroll
                            for (int p = 0; p < CH * 4; ++p) sum[p] += __builtin_bit_cast(v4f, share[j][p]);
                        }
                }
            };
            add_shares(0, split);
#pragma unroll
            for (int p = 0; p < CH * 4; ++p) {
                const v16f& x = acc[(t0 + p / 4) / TN][(t0 + p / 4) % TN];
                sum[p] += v4f{x[4 * (p % 4)], x[4 * (p % 4) + 1], x[4 * (p % 4) + 2], x[4 * (p % 4) + 3]};
            }
            add_shares(split + 1, a.splits);
#pragma unroll
            for (int t = 0; t < CH; ++t)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[(t0 + t) / TN][(t0 + t) % TN][v] = sum[t * 4 + v / 4][v % 4];
        }
    }

    // ---- epilogue ----------------------------------------------------------------------------------------------------
    // acc[i][j][v] of a lane: row (wm TM + i) 32 + lr of the tile, column (wn TN + j) 32 + 16 lg + v.  32 rows at a time go through
    // LDS so that memory sees whole rows (a lane holds 16 columns of one row: stored from there, every store would touch 64
    // lines).  Each wave has a part of LDS of its own: no barrier.
    constexpr int LPR = 4 * TN;            // lanes per row, 8 columns each
    constexpr int RPI = 64 / LPR;          // rows per pass
    constexpr int PASSES = 32 / RPI;
    constexpr int RS = TN * 32 + 4;        // floats between rows: 16 rows of one column lie in different banks
    static_assert(NW * 32 * RS * 4 <= RING, "the staging fits in the operands' LDS");
    float* const stage = reinterpret_cast<float*>(lds) + wave * (32 * RS);
    const int row0 = wm * TM * 32, col = wn * TN * 32 + (lane % LPR) * 8;
    // buffers over the tile's rows: what lies outside reads as zero and is not stored.  A column past n is marked by bits that no row
    // step clears: a tile's rows reach over less than 2^30 bytes, so the sums stay above every range and below 2^32.
    const uint32_t outside = n0 + col < a.n ? 0u : (uint32_t)kOutside;
    const __amdgpu_buffer_rsrc_t rd = make_rsrc(static_cast<uint16_t*>(a.D) + (long)m0 * a.n, (uint32_t)rows_a * (uint32_t)a.n * 2u);
    const __amdgpu_buffer_rsrc_t rbase = make_rsrc(static_cast<const uint16_t*>(a.base) + (long)m0 * a.base_stride,
                                                   a.base ? (uint32_t)((rows_a - 1) * a.base_stride + a.n) * 2u : 0u);
    const __amdgpu_buffer_rsrc_t rsa = make_rsrc(a.scale_a + (long)m0 * a.sa_stride, (uint32_t)((rows_a - 1) * a.sa_stride + 1) * 4u);
    float sb[8];
#pragma unroll
    for (int v = 0; v < 8; ++v) sb[v] = a.scale_b ? a.scale_b[(long)min(n0 + col + v, a.n - 1) * a.sb_stride] : 1.0f;
    auto write_back = [&](auto dt) __attribute__((always_inline)) {
        constexpr int DT = decltype(dt)::value;
        // The memory counter retires in order, so a load requested after stores waits for them: scales and addends of 32 rows
        // are requested before the stores of the 32 rows in front.
        v4i add[2][PASSES];
        float sa[2][PASSES];
        const uint32_t base_off = ((uint32_t)(row0 + lane / LPR) * (uint32_t)a.base_stride + (uint32_t)(n0 + col)) * 2u | outside;
        const uint32_t base_step = (uint32_t)(RPI * 2) * (uint32_t)a.base_stride;
        auto fetch = [&](int i) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < PASSES; ++r) {
                sa[i & 1][r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsa, (row0 + i * 32 + r * RPI + lane / LPR) * a.sa_stride * 4, 0, 0));
                add[i & 1][r] = __builtin_amdgcn_raw_buffer_load_b128(rbase, (int)(base_off + (uint32_t)(i * PASSES + r) * base_step), 0, 0);
            }
        };
        const uint32_t d_off = ((uint32_t)(row0 + lane / LPR) * (uint32_t)a.n + (uint32_t)(n0 + col)) * 2u | outside;
        const uint32_t d_step = (uint32_t)(RPI * 2) * (uint32_t)a.n;
        if (a.vec) fetch(0);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int p = 0; p < 4; ++p)
                    *reinterpret_cast<v4f*>(stage + lr * RS + j * 32 + lg * 16 + p * 4) =
                        v4f{acc[i][j][4 * p], acc[i][j][4 * p + 1], acc[i][j][4 * p + 2], acc[i][j][4 * p + 3]};
            if (a.vec && i + 1 < TM) fetch(i + 1);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (a.vec) {
#pragma unroll
                for (int r = 0; r < PASSES; ++r) {
                    const float* const src = stage + (r * RPI + lane / LPR) * RS + (lane % LPR) * 8;
                    const v4f x0 = reinterpret_cast<const v4f*>(src)[0], x1 = reinterpret_cast<const v4f*>(src)[1];
                    const float x[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
                    v4i o;
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const uint32_t b = (uint32_t)add[i & 1][r][v];
                        o[v] = (int)pack_pair<DT>(load16<DT>((uint16_t)(b & 0xffff)) + x[2 * v] * (sa[i & 1][r] * sb[2 * v]),
                                               load16<DT>((uint16_t)(b >> 16)) + x[2 * v + 1] * (sa[i & 1][r] * sb[2 * v + 1]));
                    }
                    __builtin_amdgcn_raw_buffer_store_b128(o, rd, (int)(d_off + (uint32_t)(i * PASSES + r) * d_step), 0, 0);
                }
            } else {  // rows of D or base that are not 16-byte aligned: one element per lane
#pragma unroll 1
                for (int e = lane; e < 32 * TN * 32; e += 64) {
                    const int r = e / (TN * 32), c = e % (TN * 32);
                    const int m = m0 + row0 + i * 32 + r, n = n0 + wn * TN * 32 + c;
                    if (m >= a.m || n >= a.n) continue;
                    float x = stage[r * RS + c] * (a.scale_a[(long)m * a.sa_stride] * (a.scale_b ? a.scale_b[(long)n * a.sb_stride] : 1.0f));
                    if (a.base) x += load16<DT>(static_cast<const uint16_t*>(a.base)[(long)m * a.base_stride + n]);
                    static_cast<uint16_t*>(a.D)[(long)m * a.n + n] = (uint16_t)pack_pair<DT>(x, 0.f);
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    };
    if (a.d_dtype == HFRK_BF16) write_back(std::integral_constant<int, HFRK_BF16>{});
    else write_back(std::integral_constant<int, HFRK_F16>{});
}

template <int TM, int TN, int WM, int WN, int NST, int WGS, bool PACKED, int LW = tiled_loader_waves(TM)>
static int launch_tiled_shape(const TiledGemmArgs& args, int lds_bytes, hipStream_t stream) {
    auto kern = tiled_gemm_kernel<TM, TN, WM, WN, NST, WGS, PACKED, LW>;
    static bool attr_done[kMaxDevices] = {};
    int dev = 0;
    HFRK_HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices || !attr_done[dev]) {
        HFRK_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes));
        if (dev >= 0 && dev < kMaxDevices) attr_done[dev] = true;
    }
    hipLaunchKernelGGL(kern, dim3(args.tiles_m * args.tiles_n * args.splits), dim3(64 * (WM * WN + LW)), lds_bytes, stream, args);
    HFRK_HIP_TRY(hipGetLastError());
    return HFRK_SUCCESS;
}

template <bool PACKED>
static int launch_tiled(const TiledGemmArgs& args, int shape, hipStream_t stream) {
    if (args.stages_q + (args.stages_r ? 1 : 0) <= 2) {
        switch (shape) {
#define HFRK_TILED_CASE(I, TM, TN, WM, WN, NST, WGS) \
    case I: return launch_tiled_shape<TM, TN, WM, WN, NST, WGS, PACKED, 0>(args, tiled_lds_bytes(kTiledShapes[I]), stream);
            HFRK_TILED_SHORT_K(HFRK_TILED_CASE)
#undef HFRK_TILED_CASE
        }
    }
    switch (shape) {
#define HFRK_TILED_CASE(I, TM, TN, WM, WN, NST, WGS) \
    case I: return launch_tiled_shape<TM, TN, WM, WN, NST, WGS, PACKED>(args, tiled_lds_bytes(kTiledShapes[I]), stream);
        HFRK_TILED_SHAPES(HFRK_TILED_CASE)
#undef HFRK_TILED_CASE
    }
    return HFRK_INVALID_CONFIG;
}

}  // namespace hfrk
