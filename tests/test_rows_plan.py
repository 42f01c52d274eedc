"""The plans that tests of the many-row forms rely on (host code: no launch)."""
import ctypes
import random

from mlx_eagle_spec_decoding_tree_amd import _lib
from test_gpu_gemm_deep import BETWEEN, SWIGLU_BETWEEN
from test_gpu_rows_builds import SHAPES, build_of


def test_the_listed_shapes_reach_every_build_that_products_pick():
    reached = {build_of(*shape) for shape in SHAPES}
    assert len(reached) == len(SHAPES)
    rng = random.Random(1)
    L = _lib.lib()
    for _ in range(60000):
        M = rng.choice([rng.randint(1, 64), rng.randint(65, 2048)])
        N, K = 8 * int(2 * 9504 ** rng.random()), 128 * int(160 ** rng.random())
        if N * K < 1 << 29 and L.eagle_qmm_rows_supported(M, N, K, 0):
            assert build_of(M, N, K) in reached, (M, N, K)


def test_rows_plan_agrees_with_the_sizes_that_callers_ask_for():
    L = _lib.lib()
    p = (ctypes.c_int * 6)()
    for M, N, K in SHAPES:
        assert L.eagle_qmm_rows_plan(M, N, K, 1, p) == 0
        assert L.eagle_qmm_rows_workspace_bytes(M, N, K) == (p[4] * M * N * 4 if p[4] > 1 else 0)
        if L.eagle_qmm_rows_plan(M, N, K, 0, p) == 0:
            assert p[4] == 1
        rc = L.eagle_qmm_rows_plan(M, N, K, 2, p)
        assert (rc == 0) == (M <= 64) and L.eagle_qmm_rows_partial_splits(M, N, K) == (p[4] if rc == 0 else 0)
    assert L.eagle_qmm_rows_plan(8, 64, 512, 1, None) == 1 and L.eagle_qmm_rows_plan(8, 64, 512, 3, p) != 0
    assert L.eagle_qmm_rows_plan(0, 64, 512, 1, p) == 2 and L.eagle_qmm_rows_plan(8, 64, 500, 1, p) == 2


def test_shapes_between_pick_the_blocks_between():
    L = _lib.lib()
    seen = set()
    for swiglu, shapes in ((0, [s[:3] for s in BETWEEN]), (1, [(M, 2 * I, K) for M, I, K in SWIGLU_BETWEEN])):
        for M, N, K in shapes:
            plan, block = (ctypes.c_int * 4)(), (ctypes.c_int * 2)()
            assert L.eagle_qmm_gemm_plan(M, N, K, swiglu, 16, 1, plan) == 0 and L.eagle_qmm_gemm_block(M, N, K, swiglu, 16, 1, block) == 0
            assert tuple(block) in ((96, 128), (160, 256), (192, 256)), (M, N, K, tuple(block))
            assert block[1] == (128 if plan[0] < 2 else 256) and plan[1] == 1
            seen.add((block[0], plan[3], plan[2] > 1, swiglu and plan[2] == 1))
    # each block with scales in fetches of four and of eight groups, split over K, whole, and whole with SwiGLU
    assert {s[:2] for s in seen} == {(r, w) for r in (96, 160, 192) for w in (4, 8)}
    assert {(s[0], s[2], s[3]) for s in seen} >= {(r, *f) for r in (96, 160, 192) for f in ((True, False), (False, 0), (False, True))}, seen


def test_gemm_block_refuses_what_the_plan_refuses():
    L = _lib.lib()
    out = (ctypes.c_int * 2)()
    assert L.eagle_qmm_gemm_block(128, 128, 128, 0, 16, 1, None) == 1
    for bad in ((0, 128, 128, 0, 16), (128, 4, 128, 0, 16), (128, 128, 100, 0, 16), (128, 128, 128, 0, 1), (128, 128, 128, 0, 6)):
        assert L.eagle_qmm_gemm_block(*bad, 1, out) == 2
