"""When a native decoder (native.py, csrc/decoder.cpp) is still the one of its model: built here on CPU tensors, which
it can be checked on but runs no pass for."""
import copy
import pickle

import pytest
import torch

from mlx_eagle_spec_decoding_tree_amd import eagle, llama, native, ops, synth

CPU = torch.device("cpu")
FUSED = dict(hidden=1024, inter=256, heads=8, kv_heads=2, head_dim=128)
PLAIN = dict(hidden=256, inter=512, heads=4, kv_heads=2, head_dim=64)


def model_of(shape, seed=3, **kw):
    args = synth.tiny(layers=2, vocab=64, attention_bias=True, **{**shape, **kw})
    return llama.Model.from_numpy(args, synth.make_model_weights(args, seed=seed), CPU)


def current(handle):
    return ops._native().decoder_current(handle)


def exchange_memory(t):
    t.data = t.data.clone()


TENSORS = {
    "gate": lambda m: m.layers[1].mlp.gate_proj.weight, "down": lambda m: m.layers[0].mlp.down_proj.scales,
    "q": lambda m: m.layers[1].self_attn.q_proj.biases, "q bias": lambda m: m.layers[0].self_attn.q_proj.bias,
    "norm": lambda m: m.layers[1].input_layernorm.weight, "last norm": lambda m: m.model.norm.weight,
    "embedding": lambda m: m.model.embed_tokens.weight, "frequencies": lambda m: m.layers[0].self_attn._inv_freqs,
}


@pytest.mark.parametrize("name", list(TENSORS))
@pytest.mark.parametrize("change", [exchange_memory, lambda t: t.mul_(1), lambda t: t.resize_(1)],
                         ids=["other memory", "counted write", "other size"])
@pytest.mark.parametrize("shape", [FUSED, PLAIN], ids=["fused", "plain"])
def test_a_decoder_is_current_until_a_tensor_changes(shape, change, name):
    model = model_of(shape)
    handle = native._build(model, "cpu")
    assert handle is not None and current(handle)
    change(TENSORS[name](model))
    assert not current(handle)


def test_exchanged_memory_stays_valid_and_its_address_is_not_taken_for_the_old_content():
    """`t.data = other` twice between two passes: the second memory cannot lie where the first lay."""
    model = model_of(FUSED)
    handle = native._build(model, "cpu")
    w = model.layers[0].mlp.gate_proj.weight
    old = w.data_ptr()
    exchange_memory(w)
    for _ in range(8):
        w.data = torch.zeros_like(w)
        assert w.data_ptr() != old
    copies = native._derive(model, *derive_args(model))
    assert copies[0] == native.FUSED and int(copies[1][0][1][0][:16].abs().max()) == 0     # layer 0, gate rows of gate|up
    assert not current(handle)


def derive_args(model):
    a = model.args
    layers = [dict(q=l.self_attn.q_proj, k=l.self_attn.k_proj, v=l.self_attn.v_proj, o=l.self_attn.o_proj,
                   gate=l.mlp.gate_proj, up=l.mlp.up_proj, down=l.mlp.down_proj) for l in model.layers]
    return layers, None, a.intermediate_size, a.hidden_size, a.num_attention_heads, a.num_key_value_heads, a.head_dim


def test_layers_of_inference_tensors_are_read_in_place():
    with torch.inference_mode():
        model = model_of(FUSED)
        for layer in model.layers:
            layer.mlp.up_proj.weight = layer.mlp.up_proj.weight.clone()
    assert native._derive(model, *derive_args(model)) == (native.PLAIN, [(None, None)] * 2)
    assert native._build(model, "cpu") is not None


def test_uncounted_writes_reach_the_copies_after_the_call_for_them():
    model = model_of(FUSED)
    form, copies = native._derive(model, *derive_args(model))
    assert form == native.FUSED
    gate = model.layers[1].mlp.gate_proj
    gate.weight.data.zero_()
    again = native._derive(model, *derive_args(model))[1]
    assert again[1][1] is copies[1][1] and int(again[1][1][0][:16].abs().max()) != 0
    model.weights_written()
    again = native._derive(model, *derive_args(model))[1]
    assert int(again[1][1][0][:16].abs().max()) == 0
    assert torch.equal(again[1][1][0], ops.interleave_gate_up(gate.weight, model.layers[1].mlp.up_proj.weight))


def test_tree_decoding_calls_a_subclass_of_the_model(monkeypatch):
    """Its own __call__, with the mask over the whole cache; a subclass without one may take the native pass."""
    class Own(llama.Model):
        def __call__(self, inputs, cache=None, mask=None, position_ids=None, flat_rope=False):
            return inputs, mask, position_ids

    class Plain(llama.Model):
        pass

    class Cache:
        offset = 5

    model, ids = model_of(PLAIN), torch.arange(3)[None]
    tree, depth = torch.zeros(3, 3), torch.arange(3)
    monkeypatch.setattr(native, "forward", lambda *a, **k: "native")
    model.__class__ = Own
    got = eagle.tree_decoding(ids, tree, depth, model, [Cache()])
    assert got[0] is ids and tuple(got[1].shape) == (1, 1, 3, 8) and got[2].tolist() == [[5, 6, 7]]
    for cls in (Plain, llama.Model):
        model.__class__ = cls
        assert eagle.tree_decoding(ids, tree, depth, model, [Cache()]) == "native"


@pytest.mark.parametrize("how", ["deepcopy", "copy", "pickle", "torch.save"])
def test_a_model_is_copied_and_stored_after_its_first_pass(how, tmp_path):
    """Without its decoder; the copy's next pass builds one on the copy's tensors."""
    model = model_of(FUSED)
    model.__dict__["_native"] = native._State(llama.Module.epoch, native._build(model, "cpu"))
    assert "_laid_out" in vars(model)
    if how == "deepcopy":
        other = copy.deepcopy(model)
    elif how == "copy":
        other = copy.copy(model)
    elif how == "pickle":
        other = pickle.loads(pickle.dumps(model))
    else:
        torch.save(model, tmp_path / "model.pt")
        other = torch.load(tmp_path / "model.pt", weights_only=False)          # written just above
    assert not any(key in vars(other) for key in native.KEPT) and all(key in vars(model) for key in native.KEPT)
    a, b = model.layers[1].mlp.up_proj.weight, other.layers[1].mlp.up_proj.weight
    assert torch.equal(a, b) and (a.data_ptr() == b.data_ptr()) == (how == "copy")
    assert current(native._build(other, "cpu")) and current(model.__dict__["_native"].handle)


@pytest.mark.parametrize("key,change", [("scales", lambda t: t.float()), ("biases", lambda t: t.float()), ("scales", lambda t: t.bfloat16()),
                                        ("scales", lambda t: t[:, :-1].contiguous()), ("biases", lambda t: t[:-1].contiguous()),
                                        ("biases", lambda t: torch.cat([t, t], 1)[:, ::2]), ("weight", lambda t: t[:-1].contiguous()),
                                        ("scales", lambda t: torch.zeros(t.numel() + 1).half()[1:].view(t.shape))])
@pytest.mark.parametrize("where", ["embedding", "head"])
@pytest.mark.parametrize("tied", [False, True], ids=["own head", "tied"])
def test_operands_of_embedding_and_head_are_checked(tied, where, key, change):
    """Types, shapes and strides that the kernels would misread leave the pass to the operators, which convert or refuse."""
    model = model_of(PLAIN, tie=tied)
    assert native._build(model, "cpu") is not None
    layer = model.model.embed_tokens if where == "embedding" or tied else model.lm_head
    setattr(layer, key, change(getattr(layer, key)))
    assert native._build(model, "cpu") is None


def test_assignments_elsewhere_do_not_rebuild_a_decoder(monkeypatch):
    """Only one that changes what the model consists of does."""
    build, built = native._build, []
    monkeypatch.setattr(native, "_build", lambda m: built.append(m) or build(m, "cpu"))
    model, other = model_of(FUSED), model_of(PLAIN)
    handle = native.decoder(model)
    assert native.decoder(model) is handle and native.decoder(other) is not None and built == [model, other]
    other.note = 1                                                 # another model, a new module, the model's own note,
    llama.RMSNorm(torch.ones(4), 1e-5)
    model.note = 2
    model.layers[0].mlp = model.layers[0].mlp                      # the same object again
    assert native.decoder(model) is handle and native.decoder(model) is handle and len(built) == 2
    up = model.layers[1].mlp.up_proj
    for change in (lambda: setattr(up, "scales", up.scales.clone()), lambda: setattr(up, "group_size", 32),
                   lambda: setattr(up, "group_size", 64), lambda: setattr(model.layers[0], "mlp", model.layers[1].mlp),
                   lambda: model.layers.reverse(), lambda: model.weights_written(),
                   lambda: setattr(model, "lm_head", llama.QuantizedLinear(up.weight, up.scales, up.biases))):
        before = len(built)
        change()
        native.decoder(model)
        assert len(built) == before + 1 and native.decoder(model) is native.decoder(model) and len(built) == before + 1


@pytest.mark.parametrize("first", ["decoder", "pass object"])
def test_decoder_and_pass_objects_share_the_laid_out_weights(first):
    """gate|up is interleaved once, and q|k|v of a pass object are row blocks that the decoder reads in place."""
    model = model_of(FUSED)
    if first == "decoder":
        assert native._build(model, "cpu") is not None
    qkv_w, gu_w = eagle.fuse_projections(model, True)
    assert "qkv" not in model.__dict__["_laid_out"]
    form, copies = native._derive(model, *derive_args(model))
    for layer, mine, (qkv, gu), fused in zip(model.layers, gu_w, copies, qkv_w):
        assert all(a.data_ptr() == b.data_ptr() for a, b in zip(gu[:3] + qkv[:3], mine[:3] + fused[:3]))
        assert qkv[0].data_ptr() == layer.self_attn.q_proj.weight.data_ptr()
        assert torch.equal(gu[0], ops.interleave_gate_up(layer.mlp.gate_proj.weight, layer.mlp.up_proj.weight))


def test_copies_go_with_the_decoder(monkeypatch):
    """Each after a wait for whoever still reads them: weights_written(), an exchanged source, a model no longer taken."""
    build, waited = native._build, []
    monkeypatch.setattr(native, "_build", lambda m: build(m, "cpu"))
    monkeypatch.setattr(native._LaidOut, "unused", lambda self: waited.append(self))
    model = model_of(FUSED)
    assert native.decoder(model) is not None
    first = dict(model.__dict__["_laid_out"])
    assert set(first) == {"qkv", "gate_up"} and not waited
    model.weights_written()
    assert sorted(map(id, waited)) == sorted(map(id, first.values())) and not model.__dict__["_laid_out"]
    assert native.decoder(model) is not None
    second = dict(model.__dict__["_laid_out"])
    exchange_memory(model.layers[0].mlp.up_proj.scales)
    native.decoder(model)
    assert waited[2:] == [second["gate_up"]] and model.__dict__["_laid_out"]["qkv"] is second["qkv"]
    model.layers[1].mlp.up_proj.group_size = 32
    assert native.decoder(model) is None and len(waited) == 5 and not model.__dict__["_laid_out"]
