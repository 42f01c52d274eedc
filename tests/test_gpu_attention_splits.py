"""Tree attention with and without key splits against 64-bit attention: every number of splits, lengths around a block of
32 keys and around the waves' deal of them, rows that see nothing, short lengths in a large cache."""
import math

import pytest
import torch

from mlx_eagle_spec_decoding_tree_amd import ops

pytestmark = pytest.mark.gpu

# scores: exact products, fp32 sums; probabilities rounded to fp16 (2^-11 relative, a 2-norm average of that over the
# keys), the result rounded to fp16: 2 * 2^-11 / sqrt(3) and some room
REL = 8e-4


def attention64(q, k, v, vis, P, Tk, scale):
    rep = q.shape[0] // k.shape[0]
    k = k[:, :P + Tk].double().repeat_interleave(rep, 0)
    v = v[:, :P + Tk].double().repeat_interleave(rep, 0)
    s = torch.matmul(q.double(), k.transpose(1, 2).contiguous()) * scale
    seen = torch.cat([torch.ones(q.shape[1], P, dtype=torch.bool, device=q.device), vis], 1)
    p = torch.nan_to_num(torch.softmax(s.masked_fill(~seen, -math.inf), -1))
    return torch.matmul(p, v).transpose(0, 1).reshape(q.shape[1], -1)


# (query heads, KV groups, head dimension): 16, 12, 8, 6, 4, 3, 2 and 1 splits at the longer caches; with 35 heads and an odd
# number of rows the partial results are an odd number of (m, l) pairs
@pytest.mark.parametrize("H,G,hd", [(2, 1, 64), (10, 2, 128), (14, 2, 64), (20, 5, 128), (28, 4, 128), (36, 9, 64),
                                    (64, 8, 128), (160, 20, 64), (1, 1, 128), (35, 5, 128)])
@pytest.mark.parametrize("cap", [64, 768, 769, 2049, 5000])
def test_splits(dev, H, G, hd, cap):
    g = torch.Generator(device=dev).manual_seed(H * 1000 + cap)
    k, v = (torch.randn(G, cap, hd, generator=g, device=dev).half() for _ in range(2))
    for T, Tk, P in ((1, 1, 0), (8, 24, 31), (8, 8, cap - 8), (32, 32, min(cap - 32, 257)), (33, 64, 0), (64, 64, cap - 64),
                     (40, 40, max(0, min(cap - 40, 2048 - 41)))):
        print(f"H={H} G={G} hd={hd} cap={cap} T={T} Tk={Tk} P={P}", flush=True)
        q = torch.randn(H, T, hd, generator=g, device=dev).half()
        vis = torch.rand(T, Tk, generator=g, device=dev) < 0.5
        if P:
            vis[0] = False
        else:
            vis[:, 0] = True
            if T > 1:
                vis[T - 1] = False             # a row that sees no key at all gives zeros
        kk, vv = k.clone(), v.clone()
        kk[:, P + Tk:], vv[:, P + Tk:] = math.nan, math.inf
        words = ops.mask_to_words(vis)
        len_dev = torch.tensor([P], dtype=torch.int32, device=dev)
        got = ops.draft_attention(q, kk, vv, words, len_dev, Tk, hd ** -0.5, max_len=cap)
        want = attention64(q, k, v, vis, P, Tk, hd ** -0.5)
        assert bool(torch.isfinite(got).all())
        assert ((got.double() - want).norm() / want.norm()).item() <= REL
        if T == Tk:
            assert torch.equal(ops.tree_attention(q, kk, vv, words, len_dev, hd ** -0.5, max_len=cap), got)
        if T > 8:                              # a row's result does not depend on the rows beside it
            few = ops.draft_attention(q[:, 3:8].contiguous(), kk, vv, words[3:8].contiguous(), len_dev, Tk, hd ** -0.5, max_len=cap)
            assert torch.equal(few, got[3:8])


# around the length from which the splits and the columns of a workgroup follow the rows, up to 32 splits, and the grid is dealt by XCD:
# groups that do and do not divide eight, fewer and more than eight, more than the division by multiplication serves
@pytest.mark.parametrize("H,G,hd", [(28, 4, 128), (32, 8, 128), (64, 8, 128), (32, 4, 64), (160, 20, 64), (1, 1, 64), (35, 5, 128),
                                    (60, 60, 64)])
@pytest.mark.parametrize("cap", [6144, 6145, 12289, 24577])
def test_long_caches(dev, H, G, hd, cap):
    g = torch.Generator(device=dev).manual_seed(H + cap)
    k, v = (torch.randn(G, cap, hd, generator=g, device=dev).half() for _ in range(2))
    for T, P in ((1, cap - 1), (1, 5), (3, 1100), (8, cap - 8), (8, 2559), (8, 5000), (16, cap - 20), (24, 3000), (32, cap - 33), (33, 4099), (64, cap - 64)):
        print(f"H={H} G={G} hd={hd} cap={cap} T={T} P={P}", flush=True)
        q = torch.randn(H, T, hd, generator=g, device=dev).half()
        vis = torch.rand(T, T, generator=g, device=dev) < 0.5
        vis[0] = False
        kk, vv = k.clone(), v.clone()
        kk[:, P + T:], vv[:, P + T:] = math.nan, math.inf
        words, len_dev = ops.mask_to_words(vis), torch.tensor([P], dtype=torch.int32, device=dev)
        # partial results of another length in the workspace: what is not in use now must not be read
        ops.draft_attention(q, k, v, words, torch.tensor([cap - T], dtype=torch.int32, device=dev), T, hd ** -0.5, max_len=cap)
        got = ops.draft_attention(q, kk, vv, words, len_dev, T, hd ** -0.5, max_len=cap)
        want = attention64(q, k, v, vis, P, T, hd ** -0.5)
        assert bool(torch.isfinite(got).all())
        assert ((got.double() - want).norm() / want.norm()).item() <= REL
        assert torch.equal(ops.tree_attention(q, kk, vv, words, len_dev, hd ** -0.5, max_len=cap), got)
