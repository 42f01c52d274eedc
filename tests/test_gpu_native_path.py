"""The native host path (csrc/host.cpp) and the kernels that came with it, against the forms they stand beside."""
import numpy as np
import pytest
import torch

from mlx_eagle_spec_decoding_tree_amd import eagle, llama, native, ops, synth
from mlx_eagle_spec_decoding_tree_amd.cache import make_prompt_cache
from oracle import tree_oracle as to
from util import MODEL_TOL, TOL, rel_err, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("root_dtype", [np.int32, np.int64])
@pytest.mark.parametrize("depth,total", [(0, 1), (0, 8), (1, 31), (1, 32), (4, 62), (5, 39), (7, 63), (15, 63)])
def test_tree_layout_from_lists(dev, depth, total, root_dtype):
    """Per-level lists read where they are, the packed retrieve rows: equal to the oracle, with frequent score ties."""
    k, rng = 8, np.random.default_rng(100 * depth + total)
    cu = np.sort(-rng.integers(0, 6, k).astype(np.float16))[::-1]
    scores, parents, chosen = [cu[None, None]], [np.zeros(1, np.int32)], np.arange(k)
    cur = cu
    for i in range(depth):
        parents.append((chosen + 1 + k * k * max(0, i - 1) + (k if i else 0)).astype(np.int32))
        c = (cur[:, None] - np.sort(rng.integers(0, 4, (k, k)), axis=1)).astype(np.float16)
        chosen = np.argsort(-c.reshape(-1).astype(np.float32), kind="stable")[:k]
        cur = c.reshape(-1)[chosen]
        scores.append(c[None])
    tokens = [rng.integers(0, 1000, s.shape).astype(np.int32) for s in scores]
    root = np.array([[7]], root_dtype)
    print(f"depth {depth} total {total}", flush=True)
    got = eagle.process_draft_tree([to_dev(s, dev) for s in scores], [to_dev(t, dev) for t in tokens],
                                   [to_dev(p, dev) for p in parents], to_dev(root, dev), k, total)
    pos, midx, toks, mask = (v.float().cpu().numpy() if v.dtype == torch.bfloat16 else v.cpu().numpy() for v in got)
    flat = [np.concatenate([v.reshape(-1) for v in part]) for part in (scores, tokens, parents)]
    dpos, dmidx, dtoks, bits = eagle.process_draft_tree_device(
        *(to_dev(v, dev) for v in flat), to_dev(root.astype(np.int32).reshape(-1), dev), k, total)
    assert np.array_equal(pos, dpos.cpu().numpy()) and np.array_equal(midx, dmidx.cpu().numpy())
    assert np.array_equal(toks, dtoks.cpu().numpy()[None]) and toks[0, 0] == 7
    assert np.array_equal(mask, eagle.bits_to_mask(bits).float().cpu().numpy())
    want = to.post_process_draft_tree(pos, total, midx)
    got = eagle.post_process_draft_tree(to_dev(pos, dev), total, to_dev(midx, dev))
    assert got.is_contiguous() and np.array_equal(got.cpu().numpy(), want)


FORMS = {       # one launch per projection; fused products, K not a multiple of 512; the same with it
    "plain": dict(hidden=256, inter=512, heads=4, kv_heads=2, head_dim=64),
    "fused": dict(hidden=896, inter=1152, heads=14, kv_heads=2, head_dim=64),
    "wide": dict(hidden=1024, inter=1536, heads=8, kv_heads=2, head_dim=128),
}


def small_model(dev, form, bias=True):
    args = synth.tiny(layers=2, vocab=1000, attention_bias=bias, **FORMS[form])
    return llama.Model.from_numpy(args, synth.make_model_weights(args, seed=3), dev)


def filled_cache(model, P, cap, seed=1):
    rng = np.random.default_rng(seed)
    cache = make_prompt_cache(model, capacity=cap)
    for c in cache:
        for buf in (c.keys, c.values):
            buf[0, :, :P] = to_dev(rng.standard_normal((buf.shape[1], P, buf.shape[3])).astype(np.float16), buf.device)
        c.offset = P
    return cache


def by_operators(model, *a, **kw):
    """The module path operator by operator."""
    keep = model.__dict__.get("_native")
    model.__dict__["_native"] = native._State(llama.Module.epoch, None)
    try:
        return model(*a, **kw)
    finally:
        model.__dict__["_native"] = keep


def same_pass(model, ids, P, cap, **kw):
    """One pass both ways; the native one must have run."""
    a, b = filled_cache(model, P, cap), filled_cache(model, P, cap)
    got = model._native_pass(ids, a, kw.get("mask"), kw.get("position_ids"), kw.get("flat_rope", False))
    assert got is not None
    want = by_operators(model, ids, b, **kw)
    assert got.shape == want.shape and a[0].offset == b[0].offset == P + ids.shape[1]
    assert rel_err(got.cpu().numpy(), want.cpu().numpy()) <= MODEL_TOL
    for x, y in zip(a, b):
        n = x.offset
        assert rel_err(x.keys[0, :, :n].cpu().numpy(), y.keys[0, :, :n].cpu().numpy()) <= MODEL_TOL
        assert rel_err(x.values[0, :, :n].cpu().numpy(), y.values[0, :, :n].cpu().numpy()) <= MODEL_TOL
    return got


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("T", [1, 16, 17, 32, 33, 64])
def test_native_tree_pass(dev, form, T):
    model, P = small_model(dev, form), 45
    rng = np.random.default_rng(T)
    depth, vis, _ = synth.tree_arrays(synth.random_tree(rng, T))
    ids = to_dev(rng.integers(0, 1000, (1, T)), dev)
    print(f"{form} T={T}", flush=True)
    mask = np.concatenate([np.zeros((T, P)), np.where(vis, 0.0, -np.inf)], axis=1).astype(np.float32)
    pos = to_dev((depth + P).astype(np.int32), dev)
    for dtype in (torch.float32, torch.bfloat16):
        got = same_pass(model, ids, P, P + T, mask=to_dev(mask, dev)[None, None].to(dtype), position_ids=pos[None])
    tree = to_dev(np.where(vis, 0.0, -np.inf).astype(np.float32), dev).to(torch.bfloat16)
    cache = filled_cache(model, P, P + T)
    again = eagle.tree_decoding(ids, tree, to_dev(depth.astype(np.int64), dev), model, cache)
    assert rel_err(again.cpu().numpy(), got.cpu().numpy()) <= MODEL_TOL and cache[1].offset == P + T


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("T,P", [(1, 0), (32, 7), (64, 0), (65, 3), (96, 40), (130, 0)])
def test_native_causal_pass(dev, form, T, P):
    model = small_model(dev, form, bias=False)
    print(f"{form} T={T} P={P}", flush=True)
    ids = to_dev(np.random.default_rng(T).integers(0, 1000, (1, T)), dev)
    same_pass(model, ids, P, P + (T + 31) // 32 * 32)
    if T <= 32:
        same_pass(model, ids, P, P + T, position_ids=5, flat_rope=True)


def test_native_decoder_follows_the_weights(dev):
    """Weights written to, exchanged layers and patched layers reach the next pass; arguments the native
    path does not take (no room for the padding of a chunk) still run."""
    model, ids = small_model(dev, "wide"), torch.arange(6, device=dev)[None]
    first = same_pass(model, ids, 3, 16)
    model.layers[1].mlp.down_proj.scales.mul_(0.5)
    second = same_pass(model, ids, 3, 16)
    assert not torch.equal(first, second)
    q = model.layers[0].self_attn.q_proj
    model.layers[0].self_attn.q_proj = llama.QuantizedLinear(q.weight, q.scales * 0.5, q.biases * 0.5, q.bias)
    third = same_pass(model, ids, 3, 16)
    assert not torch.equal(second, third)
    model.layers[0], model.layers[1] = model.layers[1], model.layers[0]
    assert not torch.equal(third, same_pass(model, ids, 3, 16))
    cache = filled_cache(model, 3, 100)
    long = torch.arange(97, device=dev)[None]
    assert model._native_pass(long, cache, None, None, False) is None and cache[0].offset == 3
    assert model(long, cache).shape == (1, 97, 1000) and cache[0].offset == 100
    llama.patch_model(model, lambda *a: ops.matmul(*a)[0])
    assert native.decoder(model) is None


def test_native_decoder_follows_memory_that_no_counter_shows(dev):
    """`t.data = other`, an uncounted write announced by weights_written(), writes to inference tensors: each reaches
    the next pass, as it does operator by operator."""
    model, ids = small_model(dev, "wide"), torch.arange(6, device=dev)[None]
    seen = [same_pass(model, ids, 3, 16)]
    for lin, key in ((model.layers[1].mlp.down_proj, "scales"), (model.layers[0].mlp.gate_proj, "weight"),
                     (model.layers[1].self_attn.q_proj, "weight"), (model.model.embed_tokens, "weight")):
        getattr(lin, key).data = getattr(lin, key).data.flip(0).contiguous()
        filler = [torch.full_like(getattr(lin, key), 0) for _ in range(4)]       # takes the old memory if it was given back
        seen.append(same_pass(model, ids, 3, 16))
        del filler
    gate = model.layers[1].mlp.gate_proj.weight
    gate.data.copy_(gate.data.flip(0))
    model.weights_written()
    seen.append(same_pass(model, ids, 3, 16))
    with torch.inference_mode():
        for layer in model.layers:
            layer.mlp.up_proj.weight = layer.mlp.up_proj.weight.clone()
        seen.append(same_pass(model, ids, 3, 16))
        up = model.layers[0].mlp.up_proj.weight
        up.copy_(up.flip(0))
        seen.append(same_pass(model, ids, 3, 16))
    assert all(not torch.equal(a, b) for i, a in enumerate(seen) for b in seen[:i] if not (i == 6 and b is seen[5]))


@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("T", [64, 65, 130, 512])
def test_a_prompt_rounds_no_weight(dev, form, T):
    """Layers that add nothing, embedding rows whose groups sum to zero, and a head of weights 64 + s q: rounded to fp16
    (multiples of 1/16) they would lose most of q, and what is left of the product is the sum of s q x."""
    args = synth.tiny(layers=1, vocab=1000, **FORMS[form])
    assert not args.tie_word_embeddings
    D, rng = args.hidden_size, np.random.default_rng(T)
    w = synth.make_model_weights(args, seed=3)
    for name in ("self_attn.o_proj", "mlp.down_proj"):
        for key in ("scales", "biases"):
            w[f"model.layers.0.{name}.{key}"][:] = 0
    q = rng.integers(0, 16, (1000, D // 2))
    nibbles = np.stack([q, 15 - q], axis=-1).reshape(1000, D // 8, 8).astype(np.uint32)
    w["model.embed_tokens.weight"] = (nibbles << (4 * np.arange(8, dtype=np.uint32))).sum(-1).astype(np.uint32)
    w["model.embed_tokens.scales"][:] = 0.25
    w["model.embed_tokens.biases"][:] = -7.5 * 0.25
    w["model.norm.weight"][:] = 1
    w["lm_head.biases"][:] = 64
    model = llama.Model.from_numpy(args, w, dev)
    ids = rng.integers(0, 1000, (1, T))
    got = model(to_dev(ids, dev), make_prompt_cache(model, capacity=T + 31))[0].cpu().numpy()
    h = (np.stack([q, 15 - q], axis=-1).reshape(1000, D) - 7.5)[ids[0]] * 0.25
    x = (h / np.sqrt((h * h).mean(1, keepdims=True) + args.rms_norm_eps)).astype(np.float16).astype(np.float64)
    words = w["lm_head.weight"]
    sq = ((words[..., None] >> (4 * np.arange(8, dtype=np.uint32))) & 15).reshape(1000, D).astype(np.float64) \
        * np.repeat(w["lm_head.scales"].astype(np.float64), 64, axis=1)
    assert rel_err(got, x @ sq.T) <= TOL


@pytest.mark.parametrize("form", ["plain", "wide"])
@pytest.mark.parametrize("T,P,spare,parts", [(2100, 3, 30, [2048, 52]), (2048 + 97, 3, 0, [2048, 64, 33]), (2049, 0, 31, [2048, 1]),
                                             (97, 3, 0, [64, 33]), (130, 0, 0, [64, 64, 2]), (96, 0, 0, [96])])
def test_long_prompts_go_in_the_largest_passes(dev, form, T, P, spare, parts, monkeypatch):
    """A prompt longer than a pass, or without room for the padding of its last one: few native calls, the bits of its parts."""
    model = small_model(dev, form)
    ids = to_dev(np.random.default_rng(T).integers(0, 1000, (1, T)), dev)
    a, b = filled_cache(model, P, P + T + spare), filled_cache(model, P, P + T + 64)
    run, taken = native.forward, []

    def counted(m, ids, *args, **kw):
        out = run(m, ids, *args, **kw)
        if out is not None:
            taken.append(ids.shape[1])
        return out

    monkeypatch.setattr(native, "forward", counted)
    got = model(ids, a)
    assert taken == parts and a[0].offset == P + T
    ends = np.cumsum(parts)
    want = torch.cat([model(ids[:, e - n:e], b) for n, e in zip(parts, ends)], dim=1)
    assert torch.equal(got, want)
    assert all(torch.equal(x.keys[:, :, :P + T], y.keys[:, :, :P + T]) for x, y in zip(a, b))


def test_the_first_pass_on_another_stream_reads_finished_copies(dev):
    """Copies laid out on a stream that is busy, then a pass on another one."""
    want = same_pass(small_model(dev, "wide"), torch.arange(6, device=dev)[None], 3, 16)
    for lay_out in (native.decoder, lambda m: eagle.fuse_projections(m, True)):
        model = small_model(dev, "wide")
        cache, ids = filled_cache(model, 3, 16), torch.arange(6, device=dev)[None]
        torch.cuda.synchronize()
        busy, other = torch.cuda.Stream(), torch.cuda.Stream()
        with torch.cuda.stream(busy):
            torch.cuda._sleep(50_000_000)
            lay_out(model)
        with torch.cuda.stream(other):
            got = model(ids, cache)
        other.synchronize()
        assert torch.equal(got, want)
