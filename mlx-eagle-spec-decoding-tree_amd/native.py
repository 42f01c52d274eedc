"""The native form of a decoder (csrc/decoder.cpp): built once per model from its layers, used by
`Model.__call__`, `tree_decoding` and the draft expansion for every pass that it takes.

A decoder is rebuilt when an attribute of a module changed, a layer was exchanged, a tensor's memory was
(`t.data = other`), or torch counted a write to a weight tensor.  A write that is not counted
(`t.data.copy_(...)`, another library on the same memory) reaches what is read in place, but not the fused
copies: after one, call `Model.weights_written()`.  Writes to inference tensors are never counted, so layers
made of them keep one launch per projection on their own tensors.  Models it does not take (a patched layer,
another group size, CPU tensors) run the Python operators of the module path."""
import torch

from . import ops
from .cache import KVCache

PLAIN, FUSED = 0, 1

# Below this hidden size the layers keep one launch per projection on the checkpoint's own tensors: their
# weights (under 4 MB per layer) are a few microseconds of reading either way, and no copy of them is made.
FUSE_HIDDEN = 768


class _State:
    """A decoder (or None: the native form does not take the model), the objects that the model then consisted of, the
    count of attribute assignments up to which it is known to consist of them, and the copies that may still be
    written."""

    def __init__(self, epoch, handle, parts=(), writing=()):
        self.epoch, self.handle, self.parts, self.writing = epoch, handle, parts, writing


def decoder(model):
    """The decoder of `model` (a handle for `forward`), or None where the native form does not take it."""
    from .llama import Module
    st = model.__dict__.get("_native")
    epoch = Module.epoch                         # (read first: an assignment meanwhile is looked for by the next pass)
    if st is not None and st.epoch != epoch:
        # something was assigned to, in this model or another: 0.1 ms for 28 layers to find out, against two for a build
        parts = _parts(model)
        if len(parts) == len(st.parts) and all(a is b for a, b in zip(parts, st.parts)):
            st.epoch = epoch
        else:
            st = None
    if st is not None and (st.handle is None or ops._native().decoder_current(st.handle)):
        if st.writing:
            st.writing = [done for done in st.writing if done.ready is not None]
            for done in st.writing:
                done.wait()
        return st.handle
    model.__dict__.pop("_native", None)          # the old decoder goes before the new one is made
    del st
    parts = _parts(model)
    handle = _build(model)
    if handle is None:
        forget(model)                            # (pass objects hold the copies that they use)
    model.__dict__["_native"] = _State(epoch, handle, parts, list(model.__dict__.get("_laid_out", {}).values()))
    return handle


def _parts(model):
    """Every attribute of the modules that a decoder is built from, in order."""
    from .llama import Module
    return ops._native().module_parts([model.args, model.model, model.__dict__.get("lm_head")], Module)


KEPT = ("_native", "_laid_out")          # what is kept with a model, and made again where it is missing


def forget(model, name=None):
    """Drop the decoder and the laid-out copies of the weights (of one name: only those); whoever needs them makes
    them again."""
    model.__dict__.pop("_native", None)
    kept = model.__dict__.get("_laid_out", {})
    for key in list(kept) if name is None else [name]:
        if key in kept:
            kept[key].unused()
            del kept[key]


def forward(model, ids, cache, mask=None, Tk=0, positions=None, pos_add=0, pos_step=0):
    """One pass (see decoder_forward in csrc/decoder.cpp): logits [1, T, V], or None where this path does not take
    the arguments (nothing has been done then)."""
    handle = decoder(model)
    if handle is None:
        return None
    return ops._native().decoder_forward(handle, ids, cache, mask, Tk, positions, pos_add, pos_step)


def _leaf(lin):
    return lin.weight, lin.scales, lin.biases, lin.bias


def _plain(w, n, k, device):
    """Whether (weight, scales, biases, bias or None) is a matrix [n, k] as the kernels read it."""
    ts = [t for t in w if t is not None]
    return (all(isinstance(t, torch.Tensor) and t.device == device and t.is_contiguous() for t in ts)
            and w[0].dtype in (torch.int32, torch.uint32) and tuple(w[0].shape) == (n, k // 8)
            and all(t.dtype == torch.float16 for t in ts[1:]) and all(t.data_ptr() % 16 == 0 for t in ts)
            and tuple(w[1].shape) == tuple(w[2].shape) == (n, k // 64) and (w[3] is None or tuple(w[3].shape) == (n,)))


def _plain_leaf(lin, n, k, device):
    from .llama import QuantizedLinear
    return type(lin) is QuantizedLinear and lin.group_size == 64 and lin.bits == 4 and _plain(_leaf(lin), n, k, device)


def _build(model, kind="cuda"):
    """The handle of a decoder on the model's tensors, which have to be on a device of this kind, or None."""
    from .llama import Attention, LlamaModel, MLP, QuantizedEmbedding, RMSNorm, TransformerBlock
    args, m = model.args, model.model
    if type(m) is not LlamaModel or not isinstance(m.layers, list) or not m.layers or type(m.norm) is not RMSNorm:
        return None
    D, I, V = args.hidden_size, args.intermediate_size, args.vocab_size
    H, G, hd = args.num_attention_heads, args.num_key_value_heads, args.head_dim
    emb = m.embed_tokens
    if type(emb) is not QuantizedEmbedding or emb.group_size != 64 or emb.bits != 4 or emb.weight.device.type != kind:
        return None
    dev = emb.weight.device
    # what the kernels of every form take
    if hd not in (64, 128) or H % G or H // G > 8 or D % 64 or I % 64 or (H * hd) % 64 or V % 8 or D > 8192:
        return None
    shapes = {"q": (H * hd, D), "k": (G * hd, D), "v": (G * hd, D), "o": (D, H * hd), "gate": (I, D), "up": (I, D),
              "down": (D, I)}
    if any(n % 8 or k % 64 for n, k in shapes.values()):
        return None
    norms = [m.norm]
    layers = []
    for layer in m.layers:
        if type(layer) is not TransformerBlock or type(layer.self_attn) is not Attention or type(layer.mlp) is not MLP:
            return None
        at, mlp = layer.self_attn, layer.mlp
        lins = dict(q=at.q_proj, k=at.k_proj, v=at.v_proj, o=at.o_proj, gate=mlp.gate_proj, up=mlp.up_proj,
                    down=mlp.down_proj)
        if not all(_plain_leaf(lin, *shapes[name], dev) for name, lin in lins.items()):
            return None
        norms += [layer.input_layernorm, layer.post_attention_layernorm]
        layers.append(lins)
    if not all(type(n) is RMSNorm and n.eps == args.rms_norm_eps and n.weight.device == dev and n.weight.dtype == torch.float16
               and n.weight.is_contiguous() and tuple(n.weight.shape) == (D,) and n.weight.data_ptr() % 16 == 0 for n in norms):
        return None
    emb_w = (emb.weight, emb.scales, emb.biases, None)
    if not _plain(emb_w, V, D, dev) or not (args.tie_word_embeddings or _plain_leaf(model.lm_head, V, D, dev)):
        return None
    head_w = emb_w if args.tie_word_embeddings else _leaf(model.lm_head)
    at0 = m.layers[0].self_attn
    if any(l.self_attn._inv_freqs is not at0._inv_freqs and not torch.equal(l.self_attn._inv_freqs, at0._inv_freqs)
           or l.self_attn._scaling_factor != at0._scaling_factor or l.self_attn.scale != at0.scale for l in m.layers):
        return None
    if at0._inv_freqs.numel() != hd // 2 or at0._inv_freqs.device != dev or at0._inv_freqs.dtype != torch.float32:
        return None

    form, derived = _derive(model, layers, shapes, I, D, H, G, hd)
    described = []
    for i, lins in enumerate(layers):
        layer = m.layers[i]
        leaves = [_leaf(lin) for lin in (layer.self_attn.q_proj, layer.self_attn.k_proj, layer.self_attn.v_proj,
                                         layer.self_attn.o_proj, layer.mlp.gate_proj, layer.mlp.up_proj, layer.mlp.down_proj)]
        described.append((*leaves, *derived[i], layer.input_layernorm.weight, layer.post_attention_layernorm.weight))
    return ops._native().decoder_new(
        (D, I, H, G, hd, V, form), (args.rms_norm_eps, float(at0._scaling_factor), float(at0.scale)), emb_w, head_w,
        m.norm.weight, at0._inv_freqs, described, m.layers, KVCache)


def _derive(model, layers, shapes, I, D, H, G, hd):
    """(form, per layer (q|k|v, gate|up))."""
    none = (None, None)
    W = (H + 2 * G) * hd
    if D < FUSE_HIDDEN or not ops.swiglu_supported(32, I, D) or W % 16 or D % 16:
        return PLAIN, [none] * len(layers)
    if any(t.is_inference() for lins in layers for name in ("q", "k", "v", "gate", "up") for t in _leaf(lins[name]) if t is not None):
        return PLAIN, [none] * len(layers)                 # a write to one could not be seen
    qkv = _lay_out(model, "qkv", _rows, [(lins["q"], lins["k"], lins["v"]) for lins in layers])
    return FUSED, list(zip(qkv, gate_up_rows(model)))


def gate_up_rows(model):
    """Per layer gate|up as `ops.interleave_gate_up` lays them out, (weight, scales, biases, bias or None): one set per
    model, for its native decoder and its pass objects."""
    return _lay_out(model, "gate_up", _gate_up, [(layer.mlp.gate_proj, layer.mlp.up_proj) for layer in model.model.layers])


def _lay_out(model, name, make, groups):
    """[make(*linears) for linears in groups], made again when a source was exchanged or torch counted a write to it."""
    leaves = [t for linears in groups for lin in linears for t in _leaf(lin) if t is not None]
    kept = model.__dict__.setdefault("_laid_out", {})
    done = kept.get(name)
    if done is None or not ops._native().sources_current(done.sources, leaves):
        done = None
        forget(model, name)                                # the old copies go before the new ones are made
        done = kept[name] = _LaidOut(ops._native().sources_new(leaves), [make(*linears) for linears in groups], leaves[0].device)
    done.wait()
    return done.copies


class _LaidOut:
    """Laid-out copies, what they were made of (its memory held with it, so that an address stands for one content), and
    until they are known to be written the event behind them."""

    def __init__(self, sources, copies, dev):
        self.sources, self.copies, self.dev = sources, copies, dev
        self.ready = torch.cuda.current_stream(dev).record_event() if dev.type == "cuda" else None

    def unused(self):
        """Returns when no stream reads the copies any more."""
        if self.dev.type == "cuda":
            torch.cuda.synchronize(self.dev)

    def wait(self):
        """Whatever the current stream enqueues from here on finds the copies written."""
        if self.ready is not None and not torch.cuda.is_current_stream_capturing():      # (a capture begins with a synchronize)
            if self.ready.query():
                self.ready = None
            else:
                torch.cuda.current_stream(self.dev).wait_event(self.ready)


def _biases(*lins):
    if all(lin.bias is None for lin in lins):
        return None
    return [lin.bias if lin.bias is not None else torch.zeros(lin.weight.shape[0], dtype=torch.float16, device=lin.weight.device)
            for lin in lins]


def _rows(*lins):
    """The matrices one below the other: a view where they already lie so, else a copy."""
    def stack(parts):
        first, at = parts[0], parts[0].data_ptr()
        for t in parts:
            if t.data_ptr() != at or t.untyped_storage().data_ptr() != first.untyped_storage().data_ptr():
                return torch.cat(parts)
            at += t.numel() * t.element_size()
        return first.as_strided((sum(t.shape[0] for t in parts), *first.shape[1:]), first.stride())
    biases = _biases(*lins)
    return (*(stack([getattr(lin, k) for lin in lins]) for k in ("weight", "scales", "biases")),
            None if biases is None else torch.cat(biases))


def _gate_up(gate, up):
    biases = _biases(gate, up)
    return (*(ops.interleave_gate_up(getattr(gate, k), getattr(up, k)) for k in ("weight", "scales", "biases")),
            None if biases is None else ops.interleave_gate_up(*biases))
