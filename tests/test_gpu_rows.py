"""The product of up to 64 rows of csrc/rows.hip, whole and split over K, plain and SwiGLU, against the oracle."""
import numpy as np
import pytest
import torch

from mlx_eagle_spec_decoding_tree_amd import _lib, ops, synth
from oracle import oracle
from util import TOL, close_fp16, layer_to_dev, rel_err, to_dev

pytestmark = pytest.mark.gpu


def call(x, d, out, swiglu, split):
    L = _lib.lib()
    M, K = x.shape
    N = d["weight"].shape[0]
    need = L.eagle_qmm_rows_workspace_bytes(M, N, K) if split else 0
    ws = torch.full((need,), 255, dtype=torch.uint8, device=x.device) if need else None
    bias = d.get("bias")
    return L.eagle_qmm_rows_w4g64_f16(x.data_ptr(), d["weight"].data_ptr(), d["scales"].data_ptr(), d["biases"].data_ptr(),
                                      bias.data_ptr() if bias is not None else None, out.data_ptr(), M, N, K, 64, 4,
                                      int(swiglu), ws.data_ptr() if need else None, need,
                                      torch.cuda.current_stream().cuda_stream)


# rows: both ends of each 16-row tile; N: less than a workgroup, no multiple of 16, several workgroups; K: less than
# a unit of four chunks, one, a remainder, many units (splits, K parts)
@pytest.mark.parametrize("M", [1, 16, 17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("N,K", [(16, 128), (24, 512), (40, 3712), (1160, 896), (904, 5248), (136, 18944), (9000, 1536)])
def test_products(dev, M, N, K):
    assert _lib.lib().eagle_qmm_rows_supported(M, N, K, 0) == 1
    print(f"rows M={M} N={N} K={K}", flush=True)
    rng = np.random.default_rng(M + N + K)
    layer = synth.make_qlinear(rng, N, K, bias=N % 16 == 8)
    x = synth.make_x(rng, M, K)
    want = oracle.qmm(x, layer["weight"], layer["scales"], layer["biases"], layer.get("bias"))
    d, xd = layer_to_dev(layer, dev), to_dev(x, dev)
    for split in (False, True):
        out = torch.full((M + 1, N), float("nan"), dtype=torch.float16, device=dev)
        rc = call(xd, d, out, False, split)
        if rc == 2 and not split and K == 18944:       # scales of this K do not fit LDS whole
            continue
        assert rc == 0
        got = out.cpu().numpy()
        assert np.isnan(got[M].astype(np.float32)).all()
        assert rel_err(got[:M], want) <= TOL, split


# divisions whose waves differ in tiles, K parts that end in one to four chunks (with one number of tiles too), a last tile of eight
# rows; rows of x at both ends of a tile
@pytest.mark.parametrize("M,N,K", [(9, 24, 1152), (9, 24, 2688), (16, 3344, 4736), (9, 6592, 4224), (2, 6624, 5248), (2, 13104, 7296), (17, 4144, 5504),
                                   (17, 6536, 4352), (32, 2360, 7168), (32, 5480, 5248), (17, 5392, 6528), (17, 8240, 3968), (32, 24, 2176),
                                   (40, 6536, 3200), (40, 8216, 3200), (48, 3272, 4864), (48, 6544, 4224), (33, 5536, 6528), (40, 8256, 3968),
                                   (48, 24, 1408), (48, 5448, 2688), (49, 6608, 3200), (64, 5544, 2688), (64, 5728, 4224), (49, 8200, 3968), (49, 48, 1152)])
def test_uneven_divisions(dev, M, N, K):
    print(f"rows M={M} N={N} K={K}", flush=True)
    rng = np.random.default_rng(M + N + K)
    for layer, x in (cancelling(rng, N, K, M), (synth.make_qlinear(rng, N, K, bias=N % 16 == 8), synth.make_x(rng, M, K))):
        d, xd = layer_to_dev(layer, dev), to_dev(x, dev)
        pick = np.unique(np.concatenate([np.arange(min(N, 40)), rng.choice(N, 300), np.arange(max(0, N - 330), N)]))
        want = oracle.qmm(x, *(layer[k][pick] for k in ("weight", "scales", "biases")), layer["bias"][pick] if "bias" in layer else None)
        for split in (False, True):
            out = torch.full((M + 1, N), float("nan"), dtype=torch.float16, device=dev)
            assert call(xd, d, out, False, split) == 0
            got = out.cpu().numpy()
            assert np.isnan(got[M].astype(np.float32)).all() and rel_err(got[:M][:, pick], want) <= TOL, split


@pytest.mark.parametrize("I,K", [(16, 896), (464, 3584), (1008, 7168), (9472, 3584), (4128, 3968)])
@pytest.mark.parametrize("M", [16, 24, 40])
def test_swiglu(dev, M, I, K):
    rng = np.random.default_rng(M + I + K)
    d = layer_to_dev(synth.make_qlinear(rng, 2 * I, K, bias=True, gain=1.0), dev)
    x = to_dev(synth.make_x(rng, M, K), dev)
    order = ops.interleave_gate_up(torch.arange(I, device=dev), torch.arange(I, 2 * I, device=dev)).long()
    inter = {k: v[order].contiguous() for k, v in d.items()}
    for split in (False, True):
        flat = torch.empty((M, 2 * I), dtype=torch.float16, device=dev)
        got = torch.empty((M, I), dtype=torch.float16, device=dev)
        assert call(x, d, flat, False, split) == 0 and call(x, inter, got, True, split) == 0
        assert torch.equal(got, ops.silu_mul(flat)), split


def test_large_head(dev):
    """Many tiles per workgroup, weight rows past the last whole workgroup."""
    M, N, K = 20, 151944, 3584
    rng = np.random.default_rng(5)
    layer = synth.make_qlinear(rng, N, K)
    x = synth.make_x(rng, M, K)
    d = layer_to_dev(layer, dev)
    got = ops.quantized_matmul(to_dev(x, dev), d["weight"], d["scales"], d["biases"]).cpu().numpy()
    rows = np.concatenate([np.arange(64), rng.choice(N, 400, replace=False), np.arange(N - 700, N)])
    want = oracle.qmm(x, layer["weight"][rows], layer["scales"][rows], layer["biases"][rows])
    assert rel_err(got[:, rows], want) <= TOL


def cancelling(rng, N, K, M):
    """Weights b + s q with b so much larger than s that fp16 would lose q, and rows of x that sum to zero in every group:
    the product is the sum of s q x, which only unrounded weights give."""
    layer = synth.make_qlinear(rng, N, K)
    layer["scales"] = rng.uniform(0.005, 0.02, (N, K // 64)).astype(np.float16)
    layer["biases"] = rng.uniform(50, 100, (N, K // 64)).astype(np.float16)
    x = rng.standard_normal((M, K // 2, 2)).astype(np.float16)
    x[..., 1] = -x[..., 0]
    return layer, x.reshape(M, K)


# rows: two blocks of 48, of 64 and less, many; N: less than a workgroup to several; K: one unit, a remainder, splits
@pytest.mark.parametrize("M,N,K", [(65, 24, 512), (96, 1160, 896), (97, 136, 18944), (130, 904, 5248), (300, 40, 3712),
                                   (1000, 264, 1536), (2047, 96, 1024), (2048, 16, 128), (129, 37888, 3584)])
def test_more_rows(dev, M, N, K):
    print(f"rows M={M} N={N} K={K}", flush=True)
    rng = np.random.default_rng(M + N + K)
    for layer, x in (cancelling(rng, N, K, M), (synth.make_qlinear(rng, N, K, bias=N % 16 == 8), synth.make_x(rng, M, K))):
        d, xd = layer_to_dev(layer, dev), to_dev(x, dev)
        pick = np.unique(np.concatenate([[0, M - 1], rng.choice(M, 22)]))
        want = oracle.qmm(x[pick], layer["weight"], layer["scales"], layer["biases"], layer.get("bias"))
        for split in (False, True):
            out = torch.full((M + 1, N), float("nan"), dtype=torch.float16, device=dev)
            rc = call(xd, d, out, False, split)
            if rc == 2 and not split and K == 18944:
                continue
            assert rc == 0
            got = out.cpu().numpy()
            assert np.isnan(got[M].astype(np.float32)).all() and rel_err(got[pick], want) <= TOL, split


@pytest.mark.parametrize("M,I,K", [(65, 16, 896), (100, 464, 3584), (2000, 48, 7168)])
def test_more_rows_with_swiglu(dev, M, I, K):
    rng = np.random.default_rng(M + I + K)
    d = layer_to_dev(synth.make_qlinear(rng, 2 * I, K, bias=True, gain=1.0), dev)
    x = to_dev(synth.make_x(rng, M, K), dev)
    order = ops.interleave_gate_up(torch.arange(I, device=dev), torch.arange(I, 2 * I, device=dev)).long()
    inter = {k: v[order].contiguous() for k, v in d.items()}
    for split in (False, True):
        flat = torch.empty((M, 2 * I), dtype=torch.float16, device=dev)
        got = torch.empty((M, I), dtype=torch.float16, device=dev)
        assert call(x, d, flat, False, split) == 0 and call(x, inter, got, True, split) == 0
        assert torch.equal(got, ops.silu_mul(flat)), split


@pytest.mark.parametrize("M", [1, 2, 17, 32])
@pytest.mark.parametrize("I,K", [(464, 3584), (48, 896), (32, 192), (4096, 512)])
def test_swiglu_of_up_to_32_rows_rounds_no_weight(dev, M, I, K):
    """The rule of ops.quantized_matmul_swiglu, with operands at its narrowest alignment too."""
    rng = np.random.default_rng(M + I + K)
    layer, x = cancelling(rng, 2 * I, K, M)
    g, u = (oracle.qmm(x, *(layer[k][h] for k in ("weight", "scales", "biases"))).astype(np.float64)
            for h in (slice(0, I), slice(I, 2 * I)))
    want = g / (1 + np.exp(-g)) * u
    d, xd = layer_to_dev(layer, dev), to_dev(x, dev)
    order = ops.interleave_gate_up(torch.arange(I, device=dev), torch.arange(I, 2 * I, device=dev)).long()
    inter = [d[k][order].contiguous() for k in ("weight", "scales", "biases")]
    for shift in (0, 1):
        sb = []
        for t in inter[1:]:
            room = torch.zeros(t.numel() + 8, dtype=torch.float16, device=dev)
            sb.append(room[shift:shift + t.numel()].view(t.shape).copy_(t))
        close_fp16(ops.quantized_matmul_swiglu(xd, inter[0], *sb).cpu().numpy(), want, f"shift {shift}", rms_frac=0.2)


@pytest.mark.parametrize("M", [33, 40, 64, 65])
@pytest.mark.parametrize("K", [192, 896, 1024])
def test_swiglu_of_more_rows_takes_any_alignment(dev, M, K):
    """Scales and biases that the slab kernel does not take go to another one."""
    I, rng = 48, np.random.default_rng(M + K)
    d = layer_to_dev(synth.make_qlinear(rng, 2 * I, K, bias=True, gain=1.0), dev)
    x = to_dev(synth.make_x(rng, M, K), dev)
    want = ops.quantized_matmul_swiglu(x, *(d[k] for k in ("weight", "scales", "biases")), bias=d["bias"]).cpu().numpy()
    room = torch.full((M + 3, I), float("nan"), dtype=torch.float16, device=dev)
    ops.quantized_matmul_swiglu(x, *(d[k] for k in ("weight", "scales", "biases")), bias=d["bias"], out=room)
    assert np.array_equal(room[:M].cpu().numpy(), want) and bool(torch.isnan(room[M:]).all())
    with pytest.raises(ValueError):
        ops.quantized_matmul_swiglu(x, *(d[k] for k in ("weight", "scales", "biases")), out=room[:M - 1])
    for shift in (1, 2, 4):
        sb = []
        for key in ("scales", "biases"):
            room = torch.zeros(d[key].numel() + 8, dtype=torch.float16, device=dev)
            sb.append(room[shift:shift + d[key].numel()].view(d[key].shape).copy_(d[key]))
        close_fp16(ops.quantized_matmul_swiglu(x, d["weight"], *sb, bias=d["bias"]).cpu().numpy(), want, f"shift {shift}", rms_frac=0.2)
