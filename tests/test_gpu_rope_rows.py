"""RoPE + K/V append where a row of the projection does not fill its workgroups: head sizes that are no power of two,
one thread short of and past a wave, one token and the most a launch takes."""
import pytest
import torch

from mlx_eagle_spec_decoding_tree_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,G,hd", [(1, 1, 16), (3, 1, 48), (6, 2, 80), (13, 1, 64), (14, 1, 64)])
@pytest.mark.parametrize("form,T", [("plain", 1), ("plain", 32), ("table", 33), ("table", 2048), ("slabs", 1), ("slabs", 64)])
def test_every_column_of_every_row(dev, H, G, hd, form, T):
    g = torch.Generator().manual_seed(H * hd + T)
    N, P, half = (H + 2 * G) * hd, 5, hd // 2
    cap = P + T + 3
    # three slabs whose sum is exact in fp32 and fp16: multiples of 1/64 below 8
    partial = (torch.randint(-160, 161, (3, ops.slab_rows(T) if T <= 64 else T, N), generator=g).float() / 64).to(dev)
    qkv = partial[:, :T].sum(0).half()
    pos = torch.randint(0, 3000, (T,), generator=g).int().to(dev)
    inv = ops.default_inv_freqs(hd, 1e4, device=dev)
    cs = ops.rope_table(pos, inv, 1.0)
    ln = torch.tensor([P], dtype=torch.int32, device=dev)
    q = torch.full((H, T, hd), 9.0, dtype=torch.float16, device=dev)
    k, v = (torch.full((G, cap, hd), 9.0, dtype=torch.float16, device=dev) for _ in range(2))
    if form == "slabs":
        ops.rope_kv_append_slabs(partial, 3, None, cs, q, k, v, ln, T, H, G, hd)
    else:
        ops.rope_kv_append(qkv, qkv[:, H * hd:], qkv[:, (H + G) * hd:], pos, inv, 1.0, q, k, v, ln, H, G, hd,
                           row_stride=N, rope_cs=cs if form == "table" else None)
    rows = qkv.double().view(T, H + 2 * G, hd).transpose(0, 1)
    angle = (inv.float()[None] * pos.float()[:, None]).double()      # the angle itself is fp32
    c, s = angle.cos(), angle.sin()
    lo, hi = rows[:H + G, :, :half], rows[:H + G, :, half:]
    want = torch.cat([lo * c - hi * s, lo * s + hi * c], -1)
    # fp16 rounding of the result, twice at most (2^-11 each), and fp32 cos, sin and products: 2^-22 of |lo| + |hi|
    bound = 2 * 2.0 ** -11 * want.abs() + 2.0 ** -22 * torch.cat([lo.abs() + hi.abs()] * 2, -1) + 2.0 ** -24
    got = torch.cat([q, k[:, P:P + T]]).double()
    assert ((got - want).abs() <= bound).all()
    assert torch.equal(v[:, P:P + T].double(), rows[H + G:])
    for cache in (k, v):
        assert (cache[:, :P] == 9).all() and (cache[:, P + T:] == 9).all()


def test_every_rotation_rounds_alike(dev):
    """The sums in fp32 on a product rounded to fp32, then fp16, bit for bit, in every kernel that rotates and in each of its elements (rounded to
    fp16 at once three in a million differ: the largest launch has nine million)."""
    g = torch.Generator().manual_seed(5)
    H, G, hd, P, half = 28, 4, 128, 3, 64
    N = (H + 2 * G) * hd
    inv = ops.default_inv_freqs(hd, 1e6, device=dev)
    ln = torch.tensor([P], dtype=torch.int32, device=dev)
    for form, T in (("table", 2048), ("plain", 32), ("slabs", 64), ("arrayed", 2048)):
        qkv = torch.randn((T, N), generator=g).half().to(dev)
        pos = (torch.arange(T) + 40).int().to(dev)
        cs = ops.rope_table(pos, inv, 1.0)
        q = torch.empty((H, T, hd), dtype=torch.float16, device=dev)
        k, v = (torch.empty((G, P + T, hd), dtype=torch.float16, device=dev) for _ in range(2))
        rows = qkv.view(T, H + 2 * G, hd).transpose(0, 1)[:H + G]
        if form == "slabs":
            partial = torch.zeros((1, ops.slab_rows(T), N), device=dev)
            partial[0, :T] = qkv.float()
            ops.rope_kv_append_slabs(partial, 1, None, cs, q, k, v, ln, T, H, G, hd)
        elif form == "arrayed":
            out = ops.arrayed_rope(rows.contiguous()[None], pos[None], inv, 1.0)[0]
            q, k[:, P:] = out[:H], out[H:]
        else:
            ops.rope_kv_append(qkv, qkv[:, H * hd:], qkv[:, (H + G) * hd:], pos, inv, 1.0, q, k, v, ln, H, G, hd, row_stride=N,
                               rope_cs=cs if form == "table" else None)
        x1, x2 = rows[..., :half].float(), rows[..., half:].float()
        co, sn = cs[..., 0], cs[..., 1]
        # (a product of 11 and 24 bits is exact in 64 bits, and so is its sum with one of 24, or rounded 29 bits below fp32)
        lo = (x1.double() * co.double() - (x2 * sn).double()).float().half()
        hi = (x1.double() * sn.double() + (x2 * co).double()).float().half()
        want = torch.cat([lo, hi], -1)
        assert torch.equal(q, want[:H]) and torch.equal(k[:, P:P + T], want[H:]), (form, int((q != want[:H]).sum()))
