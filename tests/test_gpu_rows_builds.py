"""Every build of the rows kernel that a product with a workspace picks: tiles of a wave alike and unlike in the two halves of a workgroup, one to
four tiles of x, one to four K parts, whole and half last units, one and several blocks of x.  One shape each, half of a tile in the
last weight rows, rows of x at the edges of tiles (one row in the last block of x too)."""
import ctypes

import pytest
import torch

from mlx_eagle_spec_decoding_tree_amd import _lib, ops

pytestmark = pytest.mark.gpu

SHAPES = [      # rows of x, weight rows, columns
    (1, 24, 16512), (1, 3608, 6272), (1, 24, 1152), (1, 5384, 9088), (16, 1352, 2176), (1, 6568, 3200), (1, 6552, 5248), (1, 40968, 896),
    (9, 6536, 4224), (1, 16488, 1920), (1, 12344, 6272), (1, 49224, 896), (1, 16504, 7040), (1, 65864, 896), (1, 5464, 10368), (1, 32872, 1920),
    (1, 16632, 6272), (1, 81928, 896), (1, 98360, 640), (1, 98360, 896), (17, 24, 16512), (17, 24584, 896), (17, 24, 1152), (17, 8200, 1664),
    (32, 1416, 2688), (17, 6920, 3200), (18, 8248, 3200), (17, 40968, 896), (17, 8136, 4224), (17, 16456, 1920), (17, 6920, 6272),
    (17, 49192, 896), (17, 8344, 6528), (17, 65752, 896), (17, 6184, 9088), (17, 32888, 1920), (17, 16456, 3712), (17, 81944, 384),
    (17, 8280, 14464), (17, 98328, 384), (33, 24, 16512), (33, 24600, 896), (33, 24, 1152), (48, 2696, 1664), (33, 6536, 4224), (33, 32792, 384),
    (33, 1736, 19456), (33, 16424, 1664), (33, 6936, 5248), (33, 49192, 384), (33, 8248, 6528), (33, 65544, 384), (33, 10888, 4224),
    (33, 32808, 896), (33, 16392, 3712), (33, 82008, 384), (48, 41400, 10368), (41, 41576, 9984), (33, 8280, 14592), (33, 98424, 384),
    (33, 65720, 6784), (65, 24, 16512), (65, 12296, 896), (65, 24, 1152), (129, 1400, 1664), (65, 4104, 3200), (65, 16392, 384),
    (65, 3480, 4224), (65, 8200, 896), (65, 3480, 5248), (65, 24584, 896), (65, 5384, 5248), (65, 32792, 384), (65, 16408, 1408),
    (65, 776, 19328), (65, 40968, 128), (65, 6472, 7040), (65, 20488, 1408), (65, 1448, 12928), (65, 8200, 2688), (65, 2312, 9984),
    (65, 49160, 128), (65, 8200, 13440), (65, 32776, 1408), (65, 4104, 9088), (49, 24, 16512), (49, 24, 1152), (64, 1080, 1152), (49, 24, 17024),
    (49, 32776, 640), (49, 6536, 2432), (49, 16392, 1408), (49, 3272, 4736), (49, 49160, 128), (49, 8200, 6656), (49, 65544, 128),
    (49, 8264, 9088), (49, 32824, 1408), (49, 1544, 20096), (49, 81944, 128), (49, 16408, 7296), (49, 41016, 1408), (49, 8328, 4736),
    (97, 24, 16512), (193, 264, 18560), (257, 280, 1152), (97, 24, 17024), (193, 8200, 640), (257, 136, 13440), (193, 4104, 1408),
    (257, 136, 18048), (193, 12296, 128), (193, 2056, 6528), (193, 16392, 128), (193, 2088, 9088), (193, 8216, 1408), (193, 392, 17024),
    (193, 20488, 128), (193, 4200, 7296), (193, 10248, 1408), (193, 680, 12928),
]


def build_of(M, N, K, mode=1):
    """(tiles, tiles, tiles of x, K parts, chunks of the last unit, whether x comes in blocks)"""
    p = (ctypes.c_int * 6)()
    assert _lib.lib().eagle_qmm_rows_plan(M, N, K, mode, p) == 0, (M, N, K)
    return p[0], p[1], p[2], p[3], p[5], M > 64


def product(dev, M, N, K, swiglu=False):
    """(the product by the rows kernel, weights and x in 64 bits for the weight rows `pick`, pick)"""
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (N, K // 8), dtype=torch.int32, device=dev, generator=g)
    s = (torch.rand((N, K // 64), device=dev, generator=g) * 0.02 + 0.005).half()
    b = ((torch.rand((N, K // 64), device=dev, generator=g) - 8.0) * s.float()).half()
    x = torch.randn((M, K), device=dev, generator=g).half()
    L = _lib.lib()
    need = L.eagle_qmm_rows_workspace_bytes(M, N, K)
    ws = torch.full((need,), 255, dtype=torch.uint8, device=dev)
    out = torch.full((M + 1, N // 2 if swiglu else N), float("nan"), dtype=torch.float16, device=dev)
    rc = L.eagle_qmm_rows_w4g64_f16(x.data_ptr(), w.data_ptr(), s.data_ptr(), b.data_ptr(), None, out.data_ptr(), M, N, K, 64, 4,
                                    int(swiglu), ws.data_ptr() if need else None, need, torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and bool(out[M].isnan().all())
    pick = torch.unique(torch.cat([torch.arange(min(N, 96)),
                                   torch.randint(0, N, (300,), generator=torch.Generator().manual_seed(N)), torch.arange(max(0, N - 700), N)])).to(dev)
    shift = 4 * torch.arange(8, device=dev, dtype=torch.int32)

    def wide(rows):
        q = ((w[rows][..., None] >> shift) & 15).reshape(len(rows), K).double()
        return q * s[rows].double().repeat_interleave(64, 1) + b[rows].double().repeat_interleave(64, 1)
    return out[:M], x.double(), wide, pick


# No weight is rounded: fp32 sums (of up to 20000 products, 2^-24 of partial sums some ten times the result each, independently: 1e-5) and one
# rounding to fp16, 2^-11 of the value at most.
BOUND = 2.0 ** -11 + 2e-5


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_every_build(dev, M, N, K):
    print(f"rows M={M} N={N} K={K} {build_of(M, N, K)}", flush=True)
    got, x, wide, pick = product(dev, M, N, K)
    want = x @ wide(pick).T
    err = (got[:, pick].double() - want).norm(dim=1) / want.norm(dim=1)
    assert err.max().item() <= BOUND


@pytest.mark.parametrize("M", [17, 32, 33, 40, 49, 64, 97, 128])
def test_gate_up_of_the_7b_target(dev, M):
    N, K = 37888, 3584
    got, x, wide, _ = product(dev, M, N, K, swiglu=True)
    at = torch.unique(torch.cat([torch.arange(64),
                                 torch.randint(0, N // 2, (300,), generator=torch.Generator().manual_seed(M)), torch.arange(N // 2 - 400, N // 2)])).to(dev)
    gate = at // 16 * 32 + at % 16
    g, u = x @ wide(gate).T, x @ wide(gate + 16).T
    act = torch.nn.functional.silu(g)
    # three roundings in sequence, of g, silu(g) and u; an error of g enters silu(g) times its slope, 1.1 at most; and the last one
    bound = BOUND * (1.1 * (g * u).norm() + 2 * (act * u).norm()) + 2.0 ** -11 * (act * u).norm()
    assert (got[:, at].double() - act * u).norm() <= bound
