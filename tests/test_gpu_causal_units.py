"""Attention of a prompt chunk over its divisions of the work (heads and pieces per workgroup, key splits) against 64-bit
attention: lengths around tiles of 128 keys and their halves, pieces that are not consecutive, a cache that ends with the chunk."""
import math

import pytest
import torch

from mlx_eagle_spec_decoding_tree_amd import ops

pytestmark = pytest.mark.gpu

# probabilities and the result rounded to fp16 and, with key splits, partial results too: each 2^-11 relative, averaged
# over keys and elements (2^-11 / sqrt(3) each), and some room
REL = 9e-4


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("H,G", [(1, 1), (4, 2), (6, 2), (4, 1), (5, 1), (14, 2), (28, 4), (16, 2)])
@pytest.mark.parametrize("pieces,P,spare", [(1, 0, 0), (2, 31, 0), (3, 64, 7), (5, 97, 0), (16, 0, 0), (2, 1500, 40), (9, 700, 3)])
def test_causal_chunk(dev, H, G, hd, pieces, P, spare):
    g = torch.Generator(device=dev).manual_seed(H * 100 + pieces)
    R = 32 * pieces
    cap = P + R + spare
    print(f"H={H} G={G} hd={hd} pieces={pieces} P={P} cap={cap}", flush=True)
    q = torch.randn(H, R, hd, generator=g, device=dev).half()
    k, v = (torch.randn(G, cap, hd, generator=g, device=dev).half() for _ in range(2))
    starts = P + 32 * torch.arange(pieces, device=dev)
    if pieces == 5:
        starts[3] = 5                          # a piece somewhere else in the cache
    got = ops.causal_attention(q, k, v, starts.int(), hd ** -0.5, max_len=cap)
    rows = (starts[:, None] + torch.arange(32, device=dev)[None]).reshape(-1)
    seen = torch.arange(cap, device=dev)[None] <= rows[:, None]
    want = torch.empty(R, H, hd, dtype=torch.float64, device=dev)
    for h in range(H):
        s = q[h].double() @ k[h // (H // G)].double().t().contiguous() * hd ** -0.5
        want[:, h] = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ v[h // (H // G)].double()
    want = want.reshape(R, H * hd)
    assert bool(torch.isfinite(got).all())
    assert ((got.double() - want).norm() / want.norm()).item() <= REL


@pytest.mark.parametrize("H,G,hd,R,P,value", [(16, 16, 128, 128, 16000, 20.), (32, 32, 64, 64, 16000, 20.), (28, 4, 128, 512, 32000, 20.),
                                              (14, 2, 64, 32, 5000, 32768.)])
def test_partial_results_of_long_splits(dev, H, G, hd, R, P, value):
    """A split of thousands of keys with equal scores holds thousands of times their values before they are divided by the sum of
    the probabilities.  The sums are whole numbers below 2^24 (times the value), so the result is the value itself."""
    cap = P + R
    print(f"H={H} G={G} hd={hd} R={R} P={P} value={value}", flush=True)
    q = torch.zeros(H, R, hd, device=dev).half()
    k = torch.randn(G, cap, hd, generator=torch.Generator(device=dev).manual_seed(P), device=dev).half()
    v = torch.full((G, cap, hd), value, device=dev).half()
    starts = (P + 32 * torch.arange(R // 32, device=dev)).int()
    got = ops.causal_attention(q, k, v, starts, hd ** -0.5, max_len=cap)
    assert torch.equal(got, torch.full_like(got, value))


@pytest.mark.parametrize("bad", [math.inf, math.nan])
@pytest.mark.parametrize("H,G,hd,pieces,P", [(32, 32, 64, 32, 0), (32, 32, 128, 32, 40), (16, 16, 64, 64, 1), (16, 8, 128, 64, 100), (32, 16, 64, 32, 7)])
def test_rows_of_later_pieces_stay_out(dev, H, G, hd, pieces, P, bad):
    """Fewer than four heads per group and enough pieces that a workgroup holds several: rows of the cache past a piece's end, which
    no row of it sees, may hold anything, whether they lie in a later piece or behind all of them."""
    g = torch.Generator(device=dev).manual_seed(pieces + H)
    R = 32 * pieces
    cap = P + R + 50
    print(f"H={H} G={G} hd={hd} pieces={pieces} P={P} bad={bad}", flush=True)
    q = torch.randn(H, R, hd, generator=g, device=dev).half()
    k, v = (torch.randn(G, cap, hd, generator=g, device=dev).half() for _ in range(2))
    starts = (P + 32 * torch.arange(pieces, device=dev)).int()
    want = ops.causal_attention(q, k, v, starts, hd ** -0.5, max_len=cap)
    assert bool(torch.isfinite(want).all())
    for end in (1, 2, 3, 5, pieces - 1, pieces):          # everything from the end of this many pieces on is bad
        kk, vv = k.clone(), v.clone()
        kk[:, P + 32 * end:], vv[:, P + 32 * end:] = math.nan, bad
        got = ops.causal_attention(q, kk, vv, starts, hd ** -0.5, max_len=cap)
        assert torch.equal(got[:32 * end], want[:32 * end]), end


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("H,G,pieces,P,spare", [(16, 16, 5, 1500, 0), (16, 16, 7, 3000, 5), (16, 8, 3, 5000, 0), (8, 8, 2, 9000, 3), (8, 8, 11, 700, 1),
                                                (9, 3, 3, 5000, 0), (1, 1, 1, 300, 0), (4, 2, 2, 290, 40), (16, 16, 17, 40, 0),
                                                (32, 16, 34, 30, 3000), (8, 8, 2, 50, 9000), (16, 16, 9, 4000, 0)])
def test_several_pieces_and_splits(dev, H, G, hd, pieces, P, spare):
    """Few heads per group: two, three and four pieces per workgroup, the last workgroup with fewer, and one, on split keys; splits
    that a cache much longer than the chunk leaves unused, and more than a round of workgroups."""
    test_causal_chunk(dev, H, G, hd, pieces, P, spare)
