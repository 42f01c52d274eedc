"""Slab lengths of passes above 32 rows: one round of workgroups, and the product at such lengths."""
import pytest
import torch

from mlx_eagle_spec_decoding_tree_amd import ops

CASES = [(3584, 18944), (5120, 13824), (8192, 8192), (8192, 28672), (6144, 16384), (4096, 14336), (4608, 3584), (96, 65536),
         (8192, 65536), (8192, 5120), (8200, 5120), (896, 4864)]


@pytest.mark.parametrize("M", [1, 32, 33, 40, 64])
@pytest.mark.parametrize("N,K", CASES)
def test_lengths(M, N, K):
    plain, s = ops.slab_steps(M, N, K), ops.slab_steps_one_round(M, N, K)
    if M <= 32 or plain <= 8:
        assert s == plain
        return
    groups = lambda n: (N + 127) // 128 * ops.slab_count(K, n)
    assert s >= plain and s % 8 == 0 and ops.slab_count(K, s) > 0
    assert groups(s) <= 256 or s >= K // 64
    assert s == plain or groups(s - 8) > 256             # no longer than that takes


@pytest.mark.gpu
@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("M,N,K", [(33, 3584, 18944), (40, 5120, 13824), (64, 8192, 5120), (40, 8192, 28672)])
def test_product_at_the_length_of_a_plan(dev, M, N, K, tiled):
    steps = ops.slab_steps_one_round(M, N, K)
    assert steps > ops.slab_steps(M, N, K)
    g = torch.Generator(device=dev).manual_seed(N + K)
    x = torch.randn(M, K, generator=g, device=dev).half()
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (N, K // 8), generator=g, device=dev).int()
    s = (torch.rand(N, K // 64, generator=g, device=dev) * 0.004 + 0.001).half()
    b = (-7.5 * s.float()).half()
    t = ops.tile_weights(w, s, b) if tiled else None
    got = ops.slab_sum(ops.quantized_matmul_slabs(x, w, s, b, steps, tiled=t), ops.slab_count(K, steps), M, N).double()
    rows = torch.randperm(N, generator=g, device=dev)[:64]
    shifts = torch.arange(0, 32, 4, device=dev)
    q = ((w[rows].long()[:, :, None] >> shifts) & 15).reshape(64, K).double()
    sc, bi = (v[rows].double().repeat_interleave(64, 1) for v in (s, b))
    wd = q * sc + bi
    want = x.double() @ wd.t().contiguous()
    # weights rounded to fp16 (2^-11 of each), K fp32 additions in any order (2^-24 each of the sum of magnitudes: below
    # half of the first), fp16 result
    size = x.double().abs() @ wd.abs().t().contiguous()
    # the roundings of the weights are independent: their sum has the standard deviation 2^-11 |x w|_2 / sqrt(3); six of them
    spread = (x.double() ** 2 @ (wd ** 2).t().contiguous()).sqrt()
    bound = 6 * 2.0 ** -11 * spread + 2.0 ** -24 * K ** 0.5 * size + 2.0 ** -11 * want.abs() + 1e-3
    assert ((got[:, rows] - want).abs() <= bound).all()
