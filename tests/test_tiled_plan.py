"""The tiled GEMM's planner: whatever it chooses is a plan that the entry point would accept from a caller."""
import csv
import ctypes
import os
import random

from hf_rocm_kernels import _capi

TILES = [(256, 256), (256, 128), (128, 128), (128, 64), (64, 64)]  # by shape index
WORKSPACE_BYTES = 64 << 20  # partial sums of one stream
MAX_COUNTERS = 1 << 20


def _sizes():
    rng = random.Random(1)
    # sizes whose split 256 x 256 tiles would need 97 to 128 MB
    yield from [(968, 8736, 23520), (474, 21448, 22512), (2419, 4208, 26208), (418, 16416, 26032)]
    for _ in range(20000):
        yield int(65 * 63 ** rng.random()), int(1024 * 28 ** rng.random()) // 8 * 8, int(1024 * 28 ** rng.random()) // 16 * 16


def test_partial_sums_fit_the_workspace():
    lib = _capi.load()
    for m, n, k in _sizes():
        plan = _capi.TiledPlan()
        assert lib.hfrk_tiled_gemm_plan(m, n, k, ctypes.byref(plan)) == _capi.SUCCESS
        bm, bn = TILES[plan.shape]
        tiles = -(-m // bm) * -(-n // bn)
        assert plan.splits == 1 or tiles * plan.splits * bm * bn * 4 <= WORKSPACE_BYTES, (m, n, k, plan.shape, plan.splits)
        assert plan.splits <= -(-k // 128) and 1 <= plan.group_m <= -(-m // bm)


def test_plans_of_few_rows_and_of_small_weights():
    """One row of tiles has a rule of its own, and small sizes leave few stages to split."""
    lib = _capi.load()
    rng = random.Random(2)
    sizes = [(m, n, k) for m in (1, 33, 64, 65) for n in (1, 8, 64, 65, 4104, 28672, 1 << 21) for k in (16, 128, 144, 1008, 1040, 4112, 28656)]
    sizes += [(rng.randint(1, 64), int(28672 ** rng.random()), int(1792 ** rng.random()) * 16) for _ in range(10000)]
    sizes += [(int(65 * 63 ** rng.random()), int(1024 ** rng.random()), int(64 ** rng.random()) * 16) for _ in range(10000)]
    for m, n, k in sizes:
        plan = _capi.TiledPlan()
        assert lib.hfrk_tiled_gemm_plan(m, n, k, ctypes.byref(plan)) == _capi.SUCCESS
        bm, bn = TILES[plan.shape]
        tiles, stages = -(-m // bm) * -(-n // bn), -(-k // 128)
        assert 1 <= plan.splits <= stages and 1 <= plan.group_m <= -(-m // bm), (m, n, k, plan.shape, plan.splits)
        assert plan.splits == 1 or (tiles * plan.splits * bm * bn * 4 <= WORKSPACE_BYTES and tiles <= MAX_COUNTERS and stages >= 2 * plan.splits)


def test_choices_are_those_of_the_recorded_sweep():
    """The figures beside the planner's constants are of the choices that the sweep's file marks."""
    lib = _capi.load()
    sweep = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "profiles", "tiled_gemm_plans.csv")
    measured = {}
    with open(sweep) as f:
        for row in csv.DictReader(f):
            size = tuple(int(row[x]) for x in ("m", "n", "k"))
            measured.setdefault(size, {})[int(row["shape"]), int(row["splits"])] = int(row["chosen"])
    missing = 0
    for size, plans in measured.items():
        plan = _capi.TiledPlan()
        assert lib.hfrk_tiled_gemm_plan(*size, ctypes.byref(plan)) == _capi.SUCCESS
        choice = (plan.shape, plan.splits)
        missing += choice not in plans
        assert [p for p, chosen in plans.items() if chosen] == ([choice] if choice in plans else []), size
    assert len(measured) == 260 and missing == 4  # four are split 5 ways
