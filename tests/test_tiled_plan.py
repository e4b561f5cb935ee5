"""The tiled GEMM's planner: whatever it chooses is a plan that the entry point would accept from a caller."""
import ctypes
import random

from hf_rocm_kernels import _capi

TILES = [(256, 256), (256, 128), (128, 128), (128, 64), (64, 64)]  # by shape index
WORKSPACE_BYTES = 64 << 20  # partial sums of one stream


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
