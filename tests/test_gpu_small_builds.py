"""The small-row product over its builds (one, two or four passes of x rows; one to three chunks of K per wave; ragged N)
against a 64-bit product, and SwiGLU and the folded norm on the same shapes."""
import pytest
import torch

from mlx_eagle_spec_decoding_tree_amd import ops

pytestmark = pytest.mark.gpu


def layer(dev, g, N, K):
    w = torch.randint(-2 ** 31, 2 ** 31, (N, K // 8), generator=g, device=dev, dtype=torch.int64).to(torch.int32)
    s = (torch.rand((N, K // 64), generator=g, device=dev) * 0.015 + 0.005).half()
    b = (-7.5 * s.float() + 1e-3 * torch.randn((N, K // 64), generator=g, device=dev)).half()
    q = torch.stack([(w >> (4 * i)) & 15 for i in range(8)], -1).reshape(N, K).double()
    return w, s, b, q * s.double().repeat_interleave(64, 1) + b.double().repeat_interleave(64, 1)


@pytest.mark.parametrize("K", [128, 512, 640, 896, 1024, 1152, 2048, 2944, 3584, 4864, 6144])
@pytest.mark.parametrize("T", [1, 3, 4, 5, 8, 9, 16])
def test_builds(dev, T, K):
    g = torch.Generator(device=dev).manual_seed(T * 10000 + K)
    # fp32 accumulation, a result rounded to fp16: 2^-11 / sqrt(3) of it, and the residual form's second rounding
    for N in (8, 40, 1000):
        w, s, b, full = layer(dev, g, N, K)
        x = torch.randn((T, K), generator=g, device=dev).half()
        want = x.double() @ full.t().contiguous()
        got = ops.quantized_matmul_small(x, w, s, b)
        assert ((got.double() - want).norm() / want.norm()).item() <= 4e-4, N
        res = torch.randn((T, N), generator=g, device=dev).half()
        got = ops.quantized_matmul_small(x, w, s, b, residual=res.clone())
        assert ((got.double() - want - res.double()).norm() / want.norm()).item() <= 8e-4, N
    w, s, b, full = layer(dev, g, 96, K)
    nw = (1 + 0.1 * torch.randn(K, generator=g, device=dev)).half()
    x = torch.randn((T, K), generator=g, device=dev).half() * 3
    xd = x.double()
    normed = (xd / torch.sqrt((xd * xd).mean(1, keepdim=True) + 1e-6) * nw.double()).half().double()
    pair = (normed @ full.t().contiguous()).reshape(T, 3, 2, 16)
    gate, up = pair[:, :, 0].reshape(T, 48), pair[:, :, 1].reshape(T, 48)
    want = gate / (1 + torch.exp(-gate)) * up
    got = ops.quantized_matmul_small(x, w, s, b, norm_weight=nw, eps=1e-6, swiglu=True)
    # three roundings (gate, up, silu) in sequence and that of the normalised x
    assert ((got.double() - want).norm() / want.norm()).item() <= 2e-3
