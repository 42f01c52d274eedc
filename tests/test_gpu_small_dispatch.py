"""quantized_matmul where it takes the small-row kernel: every division of K over its waves, weight rows that
are no multiple of 16, operands it does not take, against the oracle."""
import numpy as np
import pytest
import torch

from mlx_eagle_spec_decoding_tree_amd import _lib, ops, synth
from oracle import oracle
from util import TOL, layer_to_dev, rel_err, to_dev

pytestmark = pytest.mark.gpu


def run(dev, M, N, K, bias, scale=1.0):
    rng = np.random.default_rng(M + N + K)
    layer = synth.make_qlinear(rng, N, K, bias=bias)
    layer["scales"] = (layer["scales"].astype(np.float32) * scale).astype(np.float16)
    layer["biases"] = (layer["biases"].astype(np.float32) * scale).astype(np.float16)
    x = synth.make_x(rng, M, K)
    want = oracle.qmm(x, layer["weight"], layer["scales"], layer["biases"], layer.get("bias"))
    d = layer_to_dev(layer, dev)
    out = torch.full((M + 1, N), float("nan"), dtype=torch.float16, device=dev)
    ops.quantized_matmul(to_dev(x, dev), d["weight"], d["scales"], d["biases"], bias=d.get("bias"), out=out[:M])
    got = out.cpu().numpy()
    assert np.isnan(got[M].astype(np.float32)).all()
    assert rel_err(got[:M], want) <= TOL
    return d, to_dev(x, dev), got[:M]


@pytest.mark.parametrize("N,K", [(8, 128), (24, 512), (1048, 896), (96, 1024), (20480, 384), (40, 1536), (264, 2048), (8, 3072),
                                 (3592, 3584), (16, 4096), (72, 4992), (904, 6144)])
@pytest.mark.parametrize("M", [2, 8, 9, 16])
def test_products(dev, M, N, K):
    assert _lib.lib().eagle_qmm_small_preferred(M, N, K) == 1
    print(f"small M={M} N={N} K={K}", flush=True)
    run(dev, M, N, K, bias=N % 16 == 8)


def test_one_row_and_large_scales(dev):
    assert _lib.lib().eagle_qmm_small_preferred(1, 3584, 3584) == 1
    run(dev, 1, 3584, 3584, True)
    run(dev, 8, 64, 640, False, scale=200.0)           # |s| above 0.25, nibbles still exact


def test_operands_it_does_not_take(dev):
    """Scales, biases or a bias off the alignment it loads with go to another kernel, same values to the tolerance."""
    M, N, K = 5, 64, 640
    d, x, got = run(dev, M, N, K, True)
    for key in ("scales", "biases", "bias"):
        room = torch.zeros(d[key].numel() + 1, dtype=torch.float16, device=dev)
        off = room[1:].view(d[key].shape)
        off.copy_(d[key])
        e = dict(d, **{key: off})
        out = ops.quantized_matmul(x, e["weight"], e["scales"], e["biases"], bias=e["bias"])
        assert rel_err(out.cpu().numpy(), got.astype(np.float64)) <= TOL


def test_small_row_forms_take_any_alignment(dev):
    """The forms that a caller asks for by name: operands off the kernel's alignment are copied, same bits."""
    T, D, H, G, hd = 5, 256, 4, 2, 64
    W, rng = (H + 2 * G) * hd, np.random.default_rng(1)
    d = layer_to_dev(synth.make_qlinear(rng, W, D, bias=True), dev)
    x = to_dev(synth.make_x(rng, T, D), dev)

    def moved(t):
        room = torch.zeros(t.numel() + 1, dtype=torch.float16, device=dev)
        return room[1:].view(t.shape).copy_(t)

    def qkv(scales, biases, bias):
        q = torch.zeros((H, T, hd), dtype=torch.float16, device=dev)
        k, v = (torch.zeros((G, 16, hd), dtype=torch.float16, device=dev) for _ in range(2))
        ops.qkv_rope_small(x, d["weight"], scales, biases, bias, cs, q, k, v, torch.zeros(1, dtype=torch.int32, device=dev), H, G, hd)
        return torch.cat([q.flatten(), k.flatten(), v.flatten()])

    cs = ops.rope_table(torch.arange(T, dtype=torch.int32, device=dev), ops.default_inv_freqs(hd, device=dev))
    plain = [d["scales"], d["biases"], d["bias"]]
    want = ops.quantized_matmul_small(x, d["weight"], *plain[:2], bias=plain[2]), qkv(*plain)
    for i in range(3):
        e = [moved(t) if i == j else t for j, t in enumerate(plain)]
        assert torch.equal(ops.quantized_matmul_small(x, d["weight"], *e[:2], bias=e[2]), want[0])
        assert torch.equal(qkv(*e), want[1])
