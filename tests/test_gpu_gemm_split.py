"""The many-row product with K split over workgroups, against the unsplit form and the oracle."""
import numpy as np
import pytest
import torch

from mlx_eagle_spec_decoding_tree_amd import _lib, ops, synth
from oracle import oracle
from util import TOL, close_fp16, layer_to_dev, rel_err, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,bias", [(65, 8, 18944, True), (65, 200, 4864, False), (127, 904, 5184, True),
                                        (128, 3584, 3584, False), (129, 264, 9344, True), (300, 1000, 8256, False),
                                        (513, 384, 16384, True), (1000, 136, 11264, False)])
def test_split_product(dev, M, N, K, bias):
    assert _lib.lib().eagle_qmm_gemm_workspace_bytes(M, N, K, 0) > 0
    print(f"split M={M} N={N} K={K}", flush=True)
    rng = np.random.default_rng(M + N + K)
    layer = synth.make_qlinear(rng, N, K, bias=bias)
    x = synth.make_x(rng, M, K)
    d, xd = layer_to_dev(layer, dev), to_dev(x, dev)
    out = torch.full((M + 1, N), float("nan"), dtype=torch.float16, device=dev)
    ops.quantized_matmul(xd, d["weight"], d["scales"], d["biases"], bias=d.get("bias"), out=out[:M])
    got = out.cpu().numpy()
    assert np.isnan(got[M].astype(np.float32)).all()
    whole = ops.quantized_matmul(xd, d["weight"], d["scales"], d["biases"], bias=d.get("bias"), gemm=True)
    assert rel_err(got[:M], whole.cpu().numpy()) <= TOL / 2
    rows = rng.choice(M, size=24, replace=False)
    want = oracle.qmm(x[rows], layer["weight"], layer["scales"], layer["biases"], layer.get("bias"))
    assert rel_err(got[rows], want) <= TOL


@pytest.mark.parametrize("M,I,K,bias", [(65, 16, 8192, True), (100, 208, 6208, False), (129, 448, 9344, True)])
def test_split_product_with_swiglu(dev, M, I, K, bias):
    assert _lib.lib().eagle_qmm_gemm_workspace_bytes(M, 2 * I, K, 1) > 0
    print(f"split swiglu M={M} I={I} K={K}", flush=True)
    rng = np.random.default_rng(M + I + K)
    d = layer_to_dev(synth.make_qlinear(rng, 2 * I, K, bias=bias, gain=1.0), dev)
    x = to_dev(synth.make_x(rng, M, K), dev)
    args = (x, d["weight"], d["scales"], d["biases"])
    got = ops.quantized_matmul_swiglu(*args, bias=d.get("bias"))
    whole = ops.quantized_matmul_swiglu(*args, bias=d.get("bias"), gemm=True)
    close_fp16(got.cpu().numpy(), whole.cpu().numpy(), "split and whole")


@pytest.mark.parametrize("M,N,K,align,swiglu", [(513, 3584, 18944, 8, False), (129, 3584, 3584, 4, False), (81, 2304, 3584, 4, True),
                                                (130, 896, 4864, 2, False), (130, 264, 9344, 8, False)])
def test_scales_off_the_widest_alignment(dev, M, N, K, align, swiglu):
    """Scales and biases at an address that moves the split: accepted, and the product of the aligned operands."""
    print(f"M={M} N={N} K={K} align={align}", flush=True)
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (N, K // 8), dtype=torch.int32, device=dev, generator=g)
    s = (torch.rand((N, K // 64), device=dev, generator=g) * 0.004 + 0.001).half()
    b = (-7.5 * s.float()).half()
    x = torch.randn((M, K), device=dev, generator=g).half()

    def moved(t):
        room = torch.zeros(t.numel() + 8, dtype=torch.float16, device=dev)
        off = room[align // 2:align // 2 + t.numel()].view(t.shape)
        off.copy_(t)
        assert off.data_ptr() % (2 * align) == align
        return off

    op = ops.quantized_matmul_swiglu if swiglu else ops.quantized_matmul
    want = op(x, w, s, b).cpu().numpy()
    close_fp16(op(x, w, moved(s), moved(b)).cpu().numpy(), want, "moved scales")
