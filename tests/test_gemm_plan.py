"""The many-row product's workspace covers every split that its dispatch can choose (host code: no launch)."""
import ctypes

import pytest

from mlx_eagle_spec_decoding_tree_amd import _lib


def plan(M, N, K, swiglu, align, may_split=1):
    out = (ctypes.c_int * 4)()
    assert _lib.lib().eagle_qmm_gemm_plan(M, N, K, swiglu, align, may_split, out) == 0
    return tuple(out)


@pytest.mark.parametrize("swiglu", [0, 1])
@pytest.mark.parametrize("K", [64, 128, 448, 896, 3584, 4096, 4864, 5248, 9344, 14336, 18944])
def test_workspace_covers_every_alignment(K, swiglu):
    L = _lib.lib()
    for M in [65, 72, 81, 96, 100, 127, 128, 129, 200, 255, 256, 257, 300, 400, 512, 513, 700, 1000, 1024, 1025, 2047, 2048]:
        for N in (32, 64, 128, 512, 896, 1152, 2304, 3584, 4608, 9728, 18944, 37888):
            need = L.eagle_qmm_gemm_workspace_bytes(M, N, K, swiglu)
            for align in (2, 4, 8, 16):
                block, kgrp, splits, width = plan(M, N, K, swiglu, align)
                assert (splits if splits > 1 else 0) * M * N * 4 <= need, (M, N, K, align, splits)
                assert width * 2 <= align and K % (64 * width) == 0 and 0 <= block <= 3 and kgrp in (1, 2)
                assert plan(M, N, K, swiglu, align, 0)[2] == 1


def test_plan_rejects_bad_arguments():
    L = _lib.lib()
    out = (ctypes.c_int * 4)()
    assert L.eagle_qmm_gemm_plan(128, 128, 128, 0, 16, 1, None) == 1
    for bad in ((0, 128, 128, 0, 16), (128, 4, 128, 0, 16), (128, 128, 100, 0, 16), (128, 128, 128, 0, 1), (128, 128, 128, 0, 6)):
        assert L.eagle_qmm_gemm_plan(*bad, 1, out) == 2
