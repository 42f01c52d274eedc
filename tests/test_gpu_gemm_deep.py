"""The many-row product (blocks of 64 x 128 to 256 x 256, K a multiple of 256): edges of the blocks, the shortest loops,
against the product in 64 bits and the same product in passes of up to 64 rows."""
import pytest
import torch

from mlx_eagle_spec_decoding_tree_amd import ops
from util import TOL

pytestmark = pytest.mark.gpu


def layer_on(dev, N, K, bias):
    """A quantised matrix made on the device (large ones take numpy too long)."""
    g = torch.Generator(device=dev).manual_seed(N + K)
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (N, K // 8), dtype=torch.int32, device=dev, generator=g)
    s = (torch.rand((N, K // 64), device=dev, generator=g) * 0.02 + 0.005).half()
    b = (-7.5 * s.float() + 0.01 * torch.randn((N, K // 64), device=dev, generator=g)).half()
    return w, s, b, torch.randn(N, device=dev, generator=g).half() if bias else None


# Every weight is rounded to fp16 once and so is the result: each error is at most 2^-11 of its value, and errors of
# different weights do not line up, so the two together stay below sqrt(2) 2^-11 = 6.9e-4 of the result's norm.
ROUNDED = 7e-4


def product64(x, w, s, b, bias):
    q = (w[..., None] >> (4 * torch.arange(8, device=w.device, dtype=torch.int32))) & 15
    wide = lambda t: t.double().repeat_interleave(64, dim=1)  # noqa: E731
    y = x.double() @ (q.reshape(w.shape[0], -1).double() * wide(s) + wide(b)).T
    return y if bias is None else y + bias.double()


@pytest.mark.parametrize("M,N,K,bias", [(65, 8, 256, True), (129, 264, 512, False), (257, 136, 768, True), (300, 1000, 2304, False),
                                        (513, 4616, 1024, True), (2048, 4608, 512, False), (700, 18944, 256, True),
                                        (1100, 9000, 1536, False), (2047, 3592, 1280, True)])
def test_products(dev, M, N, K, bias):
    print(f"gemm M={M} N={N} K={K}", flush=True)
    w, s, b, bi = layer_on(dev, N, K, bias)
    x = torch.randn((M, K), device=dev, generator=torch.Generator(device=dev).manual_seed(M)).half()
    out = torch.full((M + 1, N), float("nan"), dtype=torch.float16, device=dev)
    ops.quantized_matmul(x, w, s, b, bias=bi, out=out[:M])
    assert torch.isnan(out[M]).all()
    want = torch.cat([ops.quantized_matmul(x[i:i + 64], w, s, b, bias=bi) for i in range(0, M, 64)]).float()
    err = (out[:M].float() - want).norm() / want.norm()
    assert err <= 1e-3 and (out[:M].float() - want).abs().amax() <= TOL * want.square().mean().sqrt()
    whole = ops.quantized_matmul(x, w, s, b, bias=bi, gemm=True).float()      # never split over K
    assert (whole - want).norm() / want.norm() <= 1e-3
    exact = product64(x, w, s, b, bi)
    for y in (out[:M], whole):
        assert (y.double() - exact).norm() / exact.norm() <= ROUNDED


@pytest.mark.parametrize("M,I,K", [(65, 16, 256), (130, 208, 512), (300, 9472, 768), (1030, 4624, 1024), (2048, 2320, 512)])
def test_swiglu(dev, M, I, K):
    w, s, b, bi = layer_on(dev, 2 * I, K, True)
    s, b = (s.float() * 0.2).half(), (b.float() * 0.2).half()
    x = torch.randn((M, K), device=dev, generator=torch.Generator(device=dev).manual_seed(M)).half()
    order = ops.interleave_gate_up(torch.arange(I, device=dev), torch.arange(I, 2 * I, device=dev)).long()
    inter = [t[order].contiguous() for t in (w, s, b, bi)]
    want = ops.silu_mul(torch.cat([ops.quantized_matmul(x[i:i + 64], w, s, b, bias=bi) for i in range(0, M, 64)])).float()
    for gemm in (None, True):
        got = ops.quantized_matmul_swiglu(x, *inter[:3], bias=inter[3], gemm=gemm).float()
        assert tuple(got.shape) == (M, I) and (got - want).norm() / want.norm() <= 2e-3
    # gate and up each within ROUNDED of their norm, silu's slope at most 1.1, and two more fp16 roundings
    g, u = product64(x, w, s, b, bi).split(I, dim=1)
    exact = torch.nn.functional.silu(g) * u
    bound = ROUNDED * (1.1 * g.norm() * u.square().mean().sqrt() + u.norm() * torch.nn.functional.silu(g).square().mean().sqrt())
    assert (got.double() - exact).norm() <= bound + 2 ** -10 * exact.norm()


# sizes whose least predicted time is that of blocks of 160, of 192 and of 96 rows: scales in fetches of four and eight groups, whole and split
# over K, the last block of rows and of columns ragged (no K of 1024: unsplit, that may be the shallow loop and its rounding)
BETWEEN = [(1738, 4616, 256, True), (1680, 4744, 512, False), (778, 1168, 7936, False), (133, 5528, 6656, True), (1937, 5272, 256, False),
           (1791, 5384, 512, True), (1608, 1200, 768, False), (908, 648, 2304, True), (1848, 1040, 512, True), (777, 592, 3584, False),
           (162, 4104, 11776, True)]
SWIGLU_BETWEEN = [(1477, 2704, 256), (1871, 2192, 512), (131, 2720, 6656), (1542, 3280, 256), (1977, 2448, 512), (1479, 656, 768),
                  (1490, 656, 512), (920, 336, 2304)]


@pytest.mark.parametrize("M,N,K,bias", BETWEEN)
def test_products_in_blocks_between(dev, M, N, K, bias):
    test_products(dev, M, N, K, bias)


@pytest.mark.parametrize("M,I,K", SWIGLU_BETWEEN)
def test_swiglu_in_blocks_between(dev, M, I, K):
    test_swiglu(dev, M, I, K)
