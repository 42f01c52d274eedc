"""quantized_matmul at both sides of the lines of the small-row kernel, the last product it takes and the first it does not, and up to
16 rows past them, where the rows kernel takes over."""
import pytest

from mlx_eagle_spec_decoding_tree_amd import _lib, ops
from test_gpu_small_dispatch import run
from util import close_fp16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,rounds", [(1, 512, 10), (1, 4096, 3), (2, 2176, 5), (4, 4992, 3), (3, 6144, 2), (5, 1536, 10), (8, 2048, 5),
                                        (8, 2560, 3), (7, 5120, 2), (9, 1024, 7), (16, 1152, 5), (16, 3584, 2), (12, 6144, 1)])
@pytest.mark.parametrize("past", [0, 8])
def test_lines(dev, M, K, rounds, past):
    N = rounds * 256 * 16 + past
    assert _lib.lib().eagle_qmm_small_preferred(M, N, K) == (past == 0)
    print(f"M={M} N={N} K={K}", flush=True)
    run(dev, M, N, K, bias=past == 0)


@pytest.mark.parametrize("M,N,K", [(2, 8200, 6144), (2, 12296, 4096), (4, 20488, 2560), (8, 20488, 2048), (16, 8200, 2048), (9, 28680, 512),
                                   (16, 24, 8192)])
def test_past_the_lines(dev, M, N, K):
    L = _lib.lib()
    assert L.eagle_qmm_rows_preferred(M, N, K) == 1 and not L.eagle_qmm_small_preferred(M, N, K) and not L.eagle_qmv_preferred(M, N, K)
    print(f"M={M} N={N} K={K}", flush=True)
    run(dev, M, N, K, bias=True)


@pytest.mark.parametrize("M,N,K", [(3, 102016, 1152), (10, 99944, 640), (4, 34496, 2816), (2, 71944, 1664), (1, 116528, 1280), (16, 99968, 640)])
def test_where_the_streaming_kernel_takes_over(dev, M, N, K):
    """The rows kernel's second round of workgroups is half empty at these numbers of weight rows."""
    L = _lib.lib()
    assert L.eagle_qmm_rows_preferred(M, N, K) == 0 and L.eagle_qmm_rows_supported(M, N, K, 0) == 1 and L.eagle_qmm_rows_preferred(M, 152064, 512) == 1
    print(f"M={M} N={N} K={K}", flush=True)
    d, x, got = run(dev, M, N, K, bias=N % 32 == 8)
    if N % 32 == 0:                                # (gate, up) tiles of 16 rows in turn
        act = ops.quantized_matmul_swiglu(x, d["weight"], d["scales"], d["biases"]).cpu().numpy()
        g, u = (got.astype("float64").reshape(M, N // 32, 2, 16)[:, :, i].reshape(M, N // 2) for i in (0, 1))
        close_fp16(act, g / (1 + 2.718281828459045 ** -g) * u)
