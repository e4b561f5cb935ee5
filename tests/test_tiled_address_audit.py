"""Address audit of the tiled GEMM on the host, no GPU: every address csrc/tiled_gemm_kernel.h forms, restated from the source for edge
tiles, first and last stages, all pieces of a stage and all lanes, and checked against what it points into (the rules are those of
test_address_audit.py: a live access lies inside its buffer, a suppressed one at or beyond its end without wrapping round)."""
import ctypes
import os
import random
import re

import numpy as np
import pytest

from hf_rocm_kernels import _capi
from test_address_audit import MAX_PANELS, U32, WS_BYTES



def _built():
    """Shape index -> the kernels built for it as (TM, TN, WM, WN, stages in LDS, waves that load), from the header that instantiates them."""
    header = os.path.join(os.path.dirname(_capi.LIB_PATH), os.pardir, "csrc", "tiled_gemm.h")
    with open(header) as f:
        lists = re.findall(r"#define HFRK_TILED_(\w+)\(X\)((?:.*\\\n)*.*)", f.read())
    built = {}
    for name, rows in lists:
        for row in re.findall(r"X\((\d), (\d), (\d), (\d), (\d), (\d), \d\)", rows):
            index, TM, TN, WM, WN, NST = map(int, row)
            built.setdefault(index, []).append((TM, TN, WM, WN, NST, 4 if TM < 4 and name != "SHORT_K" else WM * WN))
    assert sorted(built) == list(range(5)) and [len(built[i]) for i in range(5)] == [1, 3, 1, 2, 1]
    return built


BUILT = _built()
KERNELS = [(shape, kernel) for shape in sorted(BUILT) for kernel in BUILT[shape]]
KB, OUTSIDE = 128, 0x7FFFFFF0


def _half_stages(TM, NW):
    return TM * NW >= 32


def _pieces(rows, TM, NW, NL):
    """(load, wave, lane) -> row, its 16-byte piece of the stage for A and for a row-major B before the swizzle is undone, and the block of a
    packed B that a load of a stage of `rows` rows fetches."""
    q, wave = np.arange(rows * KB // (1024 * NL))[:, None, None], np.arange(NL)[None, :, None]
    if _half_stages(TM, NW):
        row = ((q >> 1) * NL + wave) * 16 + (LANE >> 2)
        swizzled = [((LANE & 3) ^ f) | (q & 1) << 2 for f in ((row >> 2) & 3, ((row >> 2) & 1) | (((row >> 4) & 1) << 1))]
        return row, *swizzled, ((q >> 1) * NL + wave) * 2 + (q & 1)
    row = (q * NL + wave) * 8 + (LANE >> 3)
    swizzled = [(LANE & 7) ^ f for f in ((row >> 1) & 7, ((row >> 1) & 3) | (((row >> 4) & 1) << 2))]
    return row, *swizzled, q * NL + wave


LANE = np.arange(64)


def _check(offsets, size, records, live, where):
    """Offsets are sums of unsigned 32-bit terms: none may reach 2^32."""
    assert (offsets >= 0).all() and (offsets + size <= U32).all(), where
    inside = offsets + size <= records
    assert (inside == live).all(), (where, "live" if (live & ~inside).any() else "suppressed")


def _edge(count):
    return sorted({0, count // 2, count - 1})


def audit(m, n, k, b_stride, plan, packed, base_stride, sa_stride=1):
    for kernel in BUILT[plan.shape]:
        _audit(kernel, m, n, k, b_stride, plan, packed, base_stride, sa_stride)


def _audit(kernel, m, n, k, b_stride, plan, packed, base_stride, sa_stride):
    TM, TN, WM, WN, NST, NL = kernel
    NW, BM, BN = WM * WN, 32 * TM * WM, 32 * TN * WN
    tiles_m, tiles_n = -(-m // BM), -(-n // BN)
    tiles, stages = tiles_m * tiles_n, -(-k // KB)
    grid = tiles * plan.splits
    ring = (BM + BN) * (KB // 2 if _half_stages(TM, NW) else KB) * NST
    assert grid * 64 * (NW + 4) < U32 and ring <= 160 * 1024

    # workgroup -> id: a bijection; tile -> (tm, tn): every tile once, whatever the group height
    per, extra = grid >> 3, grid & 7
    if grid <= 1 << 16:
        b = np.arange(grid)
        x = b & 7
        assert (np.sort(x * per + np.minimum(x, extra) + (b >> 3)) == b).all()
    if tiles <= 1 << 16:
        t = np.arange(tiles)
        group = t // (plan.group_m * tiles_n)
        in_group = t - group * plan.group_m * tiles_n
        height = np.minimum(plan.group_m, tiles_m - group * plan.group_m)
        tn = in_group // height
        tm = group * plan.group_m + in_group - tn * height
        assert (tm >= 0).all() and (tm < tiles_m).all() and (tn < tiles_n).all() and len(set(zip(tm.tolist(), tn.tolist()))) == tiles
    # stages dealt to the splits
    q, r = divmod(stages, plan.splits)
    begins = [s * q + min(s, r) for s in range(plan.splits + 1)]
    assert begins[-1] == stages and all(b > a for a, b in zip(begins, begins[1:]))

    k_tail, tail_stage = k % KB, k // KB if k % KB else -1
    for tm in _edge(tiles_m):
        m0, rows_a = tm * BM, min(BM, m - tm * BM)
        row, pa, _, _ = _pieces(BM, TM, NW, NL)
        pa = pa * 16
        assert len(np.unique(row * 8 + (pa >> 4))) == BM * 8           # every 16-byte piece of the stage is fetched once
        for s in {0, stages - 1, *(b - 1 for b in begins[1:]), *begins[:-1]}:
            records = rows_a * k - s * KB
            assert 0 < records < 1 << 31
            off = row * k + pa
            here = (row < rows_a) & (s * KB + pa < k)
            if s == tail_stage:
                off = np.where(pa < k_tail, off, OUTSIDE)
            _check(off, 16, records, here, ("A", tm, s))
            assert ((m0 + row) * k + s * KB + pa + 16 <= m * k)[here].all()
    for tn in _edge(tiles_n):
        n0 = tn * BN
        for s in {0, stages - 1, *(b - 1 for b in begins[1:]), *begins[:-1]}:
            row, _, pb, block = _pieces(BN, TM, NW, NL)
            pb = pb * 16
            if packed:
                tiles16 = min(BN // 16, (n + 15) // 16 - n0 // 16)
                t16, half, group = block >> 1, block & 1, (LANE >> 4) & 1
                slot = (LANE & 15) ^ ((t16 & 1) << 3) ^ (group << 2)
                within = (LANE >> 5) * 1024 + half * 512 + group * 256 + slot * 16
                assert len(np.unique(t16 * 128 + (within >> 4))) == BN * 8 and (within < 2048).all()
                records = tiles16 * k * 16 - s * 2048
                _check(t16 * k * 16 + within, 16, records, t16 < tiles16, ("packed B", tn, s))
                assert (n0 // 16) * k * 16 + s * 2048 + records == ((n0 // 16) + tiles16) * k * 16 <= (n + 15) // 16 * k * 16
            else:
                assert len(np.unique(row * 8 + (pb >> 4))) == BN * 8
                rows_b = min(BN, n - n0)
                records = (rows_b - 1) * b_stride + k - s * KB
                assert 0 < records < 1 << 31
                off = row * b_stride + pb
                if s == tail_stage:
                    off = np.where(pb < k_tail, off, OUTSIDE)
                _check(off, 16, records, (row < rows_b) & (s * KB + pb < k), ("B", tn, s))

    # ---- epilogue: whole rows of 8 columns a lane
    LPR = 4 * TN
    RPI = 64 // LPR
    passes = 32 // RPI
    assert NW * 32 * (TN * 32 + 4) * 4 <= ring
    for tm in _edge(tiles_m):
        m0, rows_a = tm * BM, min(BM, m - tm * BM)
        for tn in _edge(tiles_n):
            n0 = tn * BN
            for w in range(NW):
                row0, col = (w // WN) * TM * 32, (w % WN) * TN * 32 + (LANE % LPR) * 8
                outside = np.where(n0 + col < n, 0, OUTSIDE)
                step = (np.arange(TM)[:, None, None] * passes + np.arange(passes)[None, :, None])
                row = row0 + step * RPI + LANE // LPR
                if n % 8 == 0 and base_stride % 8 == 0:  # otherwise one element per lane, by indices that are compared with m and n
                    live = (row < rows_a) & (n0 + col < n)
                    d = (((row0 + LANE // LPR) * n + n0 + col) * 2 | outside) + step * (RPI * 2 * n)
                    _check(d, 16, rows_a * n * 2, live, ("D", tm, tn, w))
                    base = (((row0 + LANE // LPR) * base_stride + n0 + col) * 2 | outside) + step * (RPI * 2 * base_stride)
                    records = ((rows_a - 1) * base_stride + n) * 2
                    assert (base + 16 <= U32).all() and ((base + 16 <= records) >= live).all()
                    assert not ((base + 16 <= records) & (outside != 0)).any()
                scale = row * sa_stride * 4
                assert ((scale + 4 <= ((rows_a - 1) * sa_stride + 1) * 4) >= (row < rows_a)).all()

    # ---- partial sums
    if plan.splits > 1:
        assert tiles <= MAX_PANELS
        nmma = TM * TN
        last = ((((tiles - 1) * plan.splits + plan.splits - 1) * NW + NW - 1) * nmma + nmma - 1) * 4 + 3
        assert (last + 1) * 1024 == tiles * plan.splits * BM * BN * 4 <= WS_BYTES < 1 << 31


def test_a_turned_start_requests_every_stage_once():
    rng = random.Random(4)
    for _ in range(2000):
        begin, window, phase = rng.randint(0, 50), rng.randint(1, 43), rng.choice((0, 1, 65535, rng.randint(0, 65535)))
        end = begin + rng.randint(1, 100)
        first, last = begin, min(begin + window, end)
        left = last - first
        at, seen = first + (phase * left >> 16), []
        for _ in range(begin, end):
            assert first <= at < last
            seen.append(at)
            at = first if at + 1 == last else at + 1
            left -= 1
            if left == 0:
                first, last = last, min(last + window, end)
                left = last - first
                at = first + (phase * left >> 16)
        assert sorted(seen) == list(range(begin, end))


def _plan(m, n, k):
    plan = _capi.TiledPlan()
    assert _capi.load().hfrk_tiled_gemm_plan(m, n, k, ctypes.byref(plan)) == _capi.SUCCESS
    return plan


@pytest.mark.parametrize("shape", range(5))
@pytest.mark.parametrize("m,n,k,splits", [(1, 64, 256, 1), (64, 256, 128, 1), (257, 264, 1280, 3), (130, 203, 512, 2), (65, 136, 1008, 1),
                                          (600, 520, 768, 1), (200, 72, 16, 1), (33, 4104, 1936, 4), (70, 1032, 2064, 8), (300, 40, 784, 7)])
def test_forced_plans(shape, m, n, k, splits):
    for group_m in (1, 2):
        if group_m > -(-m // (32 * BUILT[shape][0][0] * BUILT[shape][0][2])):
            continue
        plan = _capi.TiledPlan(shape, splits, group_m)
        for base_stride in (0, n):
            audit(m, n, k, k, plan, False, base_stride)
            audit(m, n, k, k + 48, plan, False, base_stride, sa_stride=0)
        if k % 256 == 0:
            audit(m, n, k, k, plan, True, n)


def test_plans_of_the_library():
    rng = random.Random(3)
    for _ in range(60):
        m, n, k = int(33 * 125 ** rng.random()), int(8 * 3600 ** rng.random()), int(16 * 1800 ** rng.random()) // 16 * 16
        audit(m, n, k, k, _plan(m, n, k), False, n)
        k = max(256, k // 256 * 256)
        audit(m, n, k, k, _plan(m, n, k), True, 0)


@pytest.mark.parametrize("m,n,k", [(66, 1 << 21, 256), (66, (1 << 21) - 8, 16), (300, 64, 1 << 21), (1 << 24, 64, 16), (257, 1 << 21, 1 << 21)])
def test_largest_sizes(m, n, k):
    plan = _plan(m, n, k)
    for shape in range(5):
        for splits in {1, plan.splits if shape == plan.shape else 1}:
            forced = _capi.TiledPlan(shape, splits, 1)
            audit(m, n, k, 1 << 21, forced, False, n)
            audit(m, n, k, 1 << 21, forced, False, 1 << 21)
            if k % 256 == 0:
                audit(m, n, k, k, forced, True, 0)


@pytest.mark.parametrize("shape,kernel", KERNELS)
def test_every_wave_has_its_part_of_the_tile(shape, kernel):
    """The parts that the waves of a workgroup load, multiply, leave as partial sums and store are the whole tile, each once."""
    TM, TN, WM, WN, NST, NL = kernel
    NW, BM, BN = WM * WN, 32 * TM * WM, 32 * TN * WN
    assert (BM, BN) == [(256, 256), (256, 128), (128, 128), (128, 64), (64, 64)][shape]
    halves = _half_stages(TM, NW)
    stage = (BM + BN) * KB
    ring = stage * NST // 2 if halves else stage * NST
    assert ring <= 160 * 1024 and NW % 4 == 0
    loads = 0
    for rows in (BM, BN):  # A and row-major B: 8 rows of 8 pieces a load, or 16 rows of 4; packed B: half a 16-row tile's stage
        per_wave = rows * KB // (1024 * NL)
        assert per_wave * 1024 * NL == rows * KB and (not halves or per_wave % 2 == 0)
        loads += per_wave
        row, *pieces, block = _pieces(rows, TM, NW, NL)
        assert (np.sort(block.ravel()) == np.arange(rows // 8)).all()            # KB of LDS it fills
        for piece in pieces:
            assert len(np.unique(row * 8 + piece)) == rows * 8
        t16, half, group = block >> 1, block & 1, (LANE >> 4) & 1
        slot = (LANE & 15) ^ ((t16 & 1) << 3) ^ (group << 2)
        assert len(np.unique(t16 * 128 + (((LANE >> 5) * 1024 + half * 512 + group * 256 + slot * 16) >> 4))) == rows * 8
    assert (NST // 2 - 1 if halves else NST - 1) * loads <= 63                   # outstanding loads a wait can name
    # a matrix tile's rows and columns: lane lr of wave (wm, wn)
    rows = {w // WN * TM * 32 + i * 32 + lr for w in range(NW) for i in range(TM) for lr in range(32)}
    cols = {w % WN * TN * 32 + j * 32 + c for w in range(NW) for j in range(TN) for c in range(32)}
    assert rows == set(range(BM)) and cols == set(range(BN))
    # partial sums of a tile, in KB
    nmma = TM * TN
    at = {(w * nmma + t) * 4 + p for w in range(NW) for t in range(nmma) for p in range(4)}
    assert at == set(range(BM * BN * 4 // 1024))
    # epilogue: a wave's rows of 32 in LDS, then 8 columns a lane
    assert NW * 32 * (TN * 32 + 4) * 4 <= ring
    lpr = 4 * TN
    out = [(w // WN * TM * 32 + i * 32 + r * (64 // lpr) + lane // lpr, w % WN * TN * 32 + lane % lpr * 8)
           for w in range(NW) for i in range(TM) for r in range(lpr // 2) for lane in range(64)]
    assert len(out) == len(set(out)) == BM * BN // 8 and max(out) == (BM - 1, BN - 8)
