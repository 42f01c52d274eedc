// A whole pass through a decoder (mlx_llama.py:231-313 with the arguments of Model.__call__) enqueued by one
// native call: what the module path did with some thirty Python operators per layer.
//
// Bound by the host before: 30 operators x 28 layers at 10 us each, 14 ms for a 40-token tree on the 7B
// shape, whose kernels take 3 ms.  A launch from here costs about 2 us, so the GPU is the bound again.
//
// Two forms of a layer, chosen per model when the decoder is built (native.py):
//   PLAIN   one launch per projection on the checkpoint's tensors, the launches of the module path;
//   FUSED   q|k|v as one product and gate|up as one with SwiGLU in its epilogue.  Up to 16 rows, where the shapes
//           allow it, the small-row products with norm, residual, rope and cache append folded in; for 17..64 rows the
//           products stay partial sums, which the norm and rope launches add.
// No product of either form rounds a weight: more than 64 rows (a prompt) take the kernel of rows.hip in blocks and the
// causal attention, not the GEMM, which rounds every weight to fp16 (the prompt passes of spec.py use that one).  2048
// tokens on the 7B shape: 42.0 ms so, 32.1 through the GEMM, 108 in passes of 64 rows.
#include "host.h"

#include <algorithm>
#include <cmath>
#include <unordered_set>
#include <vector>

namespace eagle_host {
namespace {

enum Form { PLAIN = 0, FUSED = 1 };

struct Mat {
  const uint32_t* w = nullptr;
  const void *s = nullptr, *b = nullptr, *bias = nullptr;
  int N = 0, K = 0;
};
enum { Q, K_, V_, O, GATE, UP, DOWN, NPROJ };
struct Layer {
  Mat p[NPROJ], qkv, gu;
  const void *norm1 = nullptr, *norm2 = nullptr;
};

// A tensor that a decoder reads, as it was when the decoder was built.  The storage is held beside it: memory that
// `tensor.data = other` takes away stays valid until the decoder goes, and its address is not given out again.
struct Source {
  at::Tensor tensor;
  c10::Storage storage;
  const void* ptr;
  int64_t version;                         // (of an inference tensor: none, its writes are not counted)
  at::ScalarType type;
  at::DimVector sizes;

  // (at the implementation: seven hundred tensors are compared before a pass)
  static int64_t version_of(const at::Tensor& t) {
    const c10::VariableVersion& v = t.unsafeGetTensorImpl()->version_counter();
    return v.enabled() ? (int64_t)v.current_version() : 0;
  }
  explicit Source(const at::Tensor& t)
      : tensor(t), storage(t.storage()), ptr(t.data_ptr()), version(version_of(t)), type(t.scalar_type()), sizes(t.sizes()) {}
  bool same(const at::Tensor& now) const {
    const c10::TensorImpl* t = now.unsafeGetTensorImpl();
    return t->has_storage() && t->data() == ptr && version_of(now) == version && now.scalar_type() == type &&
           now.sizes() == sizes && now.is_contiguous();
  }
  bool same() const { return same(tensor); }
};

struct Decoder {
  int D, I, H, G, hd, V, form;
  bool linear_bias = false;                // an o or down projection with a bias
  float eps, rope_factor, scale;
  Mat emb, head;
  const void* norm = nullptr;
  const float* inv_freqs = nullptr;
  std::vector<Layer> layers;
  std::vector<Source> kept;                // every tensor whose address is held
  PyObject *layer_list = nullptr, *cache_type = nullptr;
  std::vector<PyObject*> layer_items;
};

void destroy(PyObject* cap) {
  Decoder* d = static_cast<Decoder*>(PyCapsule_GetPointer(cap, "eagle.decoder"));
  if (!d) return;
  Py_XDECREF(d->layer_list);
  Py_XDECREF(d->cache_type);
  for (PyObject* o : d->layer_items) Py_DECREF(o);
  delete d;
}

struct Bad : std::exception {
  const char* what() const noexcept override { return "unexpected decoder description"; }
};

const at::Tensor& take(Decoder* d, PyObject* o) {
  const at::Tensor* t = tensor(o);
  if (!t || !t->has_storage() || !t->is_contiguous() || (!d->kept.empty() && t->device() != d->kept[0].tensor.device())) throw Bad();
  d->kept.emplace_back(*t);
  return *t;
}
// (weight, scales, biases, bias or None)
Mat take_mat(Decoder* d, PyObject* o) {
  Mat m;
  if (o == Py_None) return m;
  if (!PyTuple_Check(o) || PyTuple_GET_SIZE(o) != 4) throw Bad();
  const at::Tensor w = take(d, PyTuple_GET_ITEM(o, 0));
  m.N = (int)w.size(0);
  m.K = (int)w.size(1) * 8;
  m.w = static_cast<const uint32_t*>(w.data_ptr());
  m.s = take(d, PyTuple_GET_ITEM(o, 1)).data_ptr();
  m.b = take(d, PyTuple_GET_ITEM(o, 2)).data_ptr();
  if (PyTuple_GET_ITEM(o, 3) != Py_None) m.bias = take(d, PyTuple_GET_ITEM(o, 3)).data_ptr();
  return m;
}
// One allocation for a pass's buffers, handed out in order
struct Arena {
  size_t size = 0;
  char* base = nullptr;
  size_t add(size_t bytes) {
    const size_t at = size;
    size += (bytes + 255) / 256 * 256;
    return at;
  }
  void* at(size_t off) const { return base + off; }
};

#define EAGLE_TRY(call)                \
  do {                                 \
    const int rc_ = (call);            \
    if (rc_ != EAGLE_OK) return rc_;   \
  } while (0)

struct Pass {
  const Decoder& d;
  const at::Tensor& like;
  void* st;
  int T, R;                              // rows, rows with padding (a prompt chunk)
  int Tk, S;                             // masked rows, rows behind the queries in all
  long cap;
  Arena ar;
  size_t h, hn, qkv, q_rot, attn, o, act, gate, down, cs, pos, words, lens, pieces, partial, attn_ws;
  size_t attn_ws_bytes = 0, partial_bytes = 0;
  int splits_qkv = 0, splits_o = 0, splits_down = 0;
  bool chunk, folded, summed, fused;
  std::vector<void*> keys, values;

  void* p(size_t off) const { return ar.at(off); }
  int* len(int i) const { return static_cast<int*>(p(lens)) + i; }

  void plan() {
    const int W = (d.H + 2 * d.G) * d.hd;
    chunk = T > 2 * EAGLE_MAX_TREE;
    fused = d.form == FUSED;
    folded = fused && T <= 16 && eagle_qkv_rope_small_supported(T, d.D, d.H, d.G, d.hd) &&
             eagle_qmm_small_supported(T, d.D, d.H * d.hd, 0, 0) && eagle_qmm_small_supported(T, 2 * d.I, d.D, 1, 1) &&
             eagle_qmm_small_supported(T, d.D, d.I, 0, 0);
    summed = false;
    if (fused && !chunk && T > EAGLE_MAX_M / 2 && !d.linear_bias) {
      splits_qkv = eagle_qmm_rows_partial_splits(T, W, d.D);
      splits_o = eagle_qmm_rows_partial_splits(T, d.D, d.H * d.hd);
      splits_down = eagle_qmm_rows_partial_splits(T, d.D, d.I);
      summed = splits_qkv && splits_o && splits_down;
      const size_t rows = T > EAGLE_MAX_M ? 2 * EAGLE_MAX_M : EAGLE_MAX_M;
      partial_bytes = summed ? rows * sizeof(float) * std::max({(size_t)splits_qkv * W, (size_t)splits_o * d.D, (size_t)splits_down * d.D}) : 0;
    }
    const size_t f16 = 2, rows = (size_t)R;
    h = ar.add(rows * d.D * f16);
    hn = ar.add(rows * d.D * f16);
    qkv = ar.add(rows * W * f16);
    q_rot = ar.add(rows * d.H * d.hd * f16);
    attn = ar.add(rows * d.H * d.hd * f16);
    o = ar.add(rows * d.D * f16);
    act = ar.add(rows * d.I * f16);
    gate = ar.add(d.form == FUSED ? 256 : rows * 2 * d.I * f16);
    cs = ar.add(rows * (d.hd / 2) * 2 * 4);
    pos = ar.add(rows * 4);
    words = ar.add(rows * 2 * 4);
    lens = ar.add(8);
    pieces = ar.add((rows / 32 + 1) * 4);
    partial = ar.add(partial_bytes);
    attn_ws_bytes = chunk ? eagle_causal_attention_workspace_bytes(R, d.H, d.hd, S)
                          : eagle_tree_attention_wide_workspace_bytes(T, d.H, d.hd, S);
    attn_ws = ar.add(attn_ws_bytes);
  }

  // more than 64 rows without rounding a weight: in blocks by one launch, or where that kernel does not take the operands
  // in passes of 64
  int product(const Mat& m, const void* x, void* out, int M) {
    constexpr int PASS = 2 * EAGLE_MAX_M;
    if (M <= PASS) return matmul(like, x, m.w, m.s, m.b, m.bias, out, M, m.N, m.K, st);
    if (eagle_qmm_rows_supported(M, m.N, m.K, 0) && small_aligned(x, m.s, m.b, nullptr, out))
      return rows(like, x, m.w, m.s, m.b, m.bias, out, M, m.N, m.K, false, st);
    for (int r0 = 0; r0 < M; r0 += PASS)
      EAGLE_TRY(product(m, static_cast<const char*>(x) + (size_t)r0 * m.K * 2, static_cast<char*>(out) + (size_t)r0 * m.N * 2,
                        std::min(M - r0, PASS)));
    return EAGLE_OK;
  }
  int product(const Mat& m, const void* x, void* out) { return product(m, x, out, R); }

  int attention(int i) {
    if (chunk)
      return eagle_causal_attention_f16(p(q_rot), keys[i], values[i], static_cast<const int32_t*>(p(pieces)), p(attn), R, d.H,
                                        d.G, d.hd, cap, S, d.scale, p(attn_ws), attn_ws_bytes, st);
    const uint32_t* m = static_cast<const uint32_t*>(p(words));
    if (T > EAGLE_MAX_TREE)
      return eagle_tree_attention_wide_f16(p(q_rot), keys[i], values[i], m, len(1), p(attn), T, Tk, d.H, d.G, d.hd, cap, S,
                                           d.scale, p(attn_ws), attn_ws_bytes, st);
    return eagle_draft_attention_f16(p(q_rot), keys[i], values[i], m, len(1), p(attn), T, Tk, d.H, d.G, d.hd, cap, S, d.scale,
                                     p(attn_ws), attn_ws_bytes, st);
  }

  int partial_product(const Mat& m, const void* x) {
    return eagle_qmm_rows_partial_w4g64(x, m.w, m.s, m.b, static_cast<float*>(p(partial)), partial_bytes, T, m.N, m.K, 64, 4, st);
  }

  int layer(int i, const void* next_norm) {
    const Layer& l = d.layers[i];
    const float* part = static_cast<const float*>(p(partial));
    const float* table = static_cast<const float*>(p(cs));
    const int W = (d.H + 2 * d.G) * d.hd;
    if (folded) {
      EAGLE_TRY(eagle_qkv_rope_small_w4g64_f16(p(h), l.norm1, d.eps, l.qkv.w, l.qkv.s, l.qkv.b, l.qkv.bias, table, p(q_rot), keys[i],
                                               values[i], len(0), T, d.D, d.H, d.G, d.hd, cap, 64, 4, st));
      EAGLE_TRY(attention(i));
      const Mat &mo = l.p[O], &md = l.p[DOWN];
      EAGLE_TRY(eagle_qmm_small_w4g64_f16(p(attn), nullptr, d.eps, mo.w, mo.s, mo.b, mo.bias, p(h), p(h), T, mo.N, mo.K, 64, 4, 0, st));
      EAGLE_TRY(eagle_qmm_small_w4g64_f16(p(h), l.norm2, d.eps, l.gu.w, l.gu.s, l.gu.b, l.gu.bias, nullptr, p(act), T, l.gu.N,
                                          l.gu.K, 64, 4, 1, st));
      return eagle_qmm_small_w4g64_f16(p(act), nullptr, d.eps, md.w, md.s, md.b, md.bias, p(h), p(h), T, md.N, md.K, 64, 4, 0, st);
    }
    if (summed) {
      EAGLE_TRY(partial_product(l.qkv, p(hn)));
      EAGLE_TRY(eagle_rope_kv_append_slabs_f16(part, splits_qkv, l.qkv.bias, table, p(q_rot), keys[i], values[i], len(0), T, d.H, d.G,
                                               d.hd, cap, st));
    } else if (fused) {
      EAGLE_TRY(product(l.qkv, p(hn), p(qkv)));
      const char* base = static_cast<const char*>(p(qkv));
      EAGLE_TRY(eagle_rope_kv_append_table_f16(base, base + (size_t)d.H * d.hd * 2, base + (size_t)(d.H + d.G) * d.hd * 2, table,
                                               p(q_rot), keys[i], values[i], len(0), R, d.H, d.G, d.hd, cap, W, st));
    } else {
      char* q = static_cast<char*>(p(qkv));
      char* k = q + (size_t)R * d.H * d.hd * 2;
      char* v = k + (size_t)R * d.G * d.hd * 2;
      EAGLE_TRY(product(l.p[Q], p(hn), q));
      EAGLE_TRY(product(l.p[K_], p(hn), k));
      EAGLE_TRY(product(l.p[V_], p(hn), v));
      if (R <= EAGLE_MAX_TREE)
        EAGLE_TRY(eagle_rope_kv_append_f16(q, k, v, static_cast<const int32_t*>(p(pos)), d.inv_freqs, d.rope_factor, p(q_rot),
                                           keys[i], values[i], len(0), R, d.H, d.G, d.hd, cap, 0, st));
      else
        EAGLE_TRY(eagle_rope_kv_append_table_f16(q, k, v, table, p(q_rot), keys[i], values[i], len(0), R, d.H, d.G, d.hd, cap, 0,
                                                 st));
    }
    EAGLE_TRY(attention(i));
    if (summed) {
      EAGLE_TRY(partial_product(l.p[O], p(attn)));
      EAGLE_TRY(eagle_rmsnorm_slabs_f16(part, splits_o, p(h), l.norm2, d.eps, p(h), p(hn), T, d.D, st));
      EAGLE_TRY(swiglu(like, p(hn), l.gu.w, l.gu.s, l.gu.b, l.gu.bias, p(act), R, l.gu.N, l.gu.K, true, st));
      EAGLE_TRY(partial_product(l.p[DOWN], p(act)));
      return eagle_rmsnorm_slabs_f16(part, splits_down, p(h), next_norm, d.eps, p(h), p(hn), T, d.D, st);
    }
    EAGLE_TRY(product(l.p[O], p(attn), p(o)));
    EAGLE_TRY(eagle_rmsnorm_f16(p(o), p(h), l.norm2, d.eps, p(h), p(hn), R, d.D, st));
    if (fused) {
      EAGLE_TRY(swiglu(like, p(hn), l.gu.w, l.gu.s, l.gu.b, l.gu.bias, p(act), R, l.gu.N, l.gu.K, true, st));
    } else {
      char* up = static_cast<char*>(p(gate)) + (size_t)R * d.I * 2;
      EAGLE_TRY(product(l.p[GATE], p(hn), p(gate)));
      EAGLE_TRY(product(l.p[UP], p(hn), up));
      EAGLE_TRY(eagle_silu_mul_f16(p(gate), up, p(act), R, d.I, st));
    }
    EAGLE_TRY(product(l.p[DOWN], p(act), p(o)));
    return eagle_rmsnorm_f16(p(o), p(h), next_norm, d.eps, p(h), p(hn), R, d.D, st);
  }
};

PyObject* str(const char* s) { return PyUnicode_InternFromString(s); }

}  // namespace

// The tensors of a list as they are now
static bool list_sources(PyObject* list, std::vector<const at::Tensor*>* out) {
  if (!PyList_Check(list)) return false;
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(list); ++i) {
    out->push_back(tensor(PyList_GET_ITEM(list, i)));
    if (!out->back() || !out->back()->has_storage()) return false;
  }
  return true;
}

// module_parts(roots, Module) -> every attribute of the modules among `roots` and of those they hold, in order (a few
// thousand objects, 30 us; a walk in Python takes ten times that)
PyObject* py_module_parts(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 2 || !PyList_Check(a[0]) || !PyType_Check(a[1])) {
    PyErr_SetString(PyExc_TypeError, "module_parts takes a list and a type");
    return nullptr;
  }
  PyTypeObject* type = reinterpret_cast<PyTypeObject*>(a[1]);
  PyObject* found = PyList_GetSlice(a[0], 0, PyList_GET_SIZE(a[0]));
  std::vector<PyObject*> todo;                       // (all held by `found` or by the roots)
  std::unordered_set<PyObject*> seen;
  auto look = [&](PyObject* o) {
    if (PyObject_TypeCheck(o, type)) todo.push_back(o);
  };
  for (Py_ssize_t i = 0; found && i < PyList_GET_SIZE(found); ++i) look(PyList_GET_ITEM(found, i));
  while (found && !todo.empty()) {
    PyObject* m = todo.back();
    todo.pop_back();
    if (!seen.insert(m).second) continue;
    PyObject* dict = PyObject_GenericGetDict(m, nullptr);
    PyObject *key, *value;
    Py_ssize_t at = 0;
    bool ok = dict != nullptr;
    while (ok && PyDict_Next(dict, &at, &key, &value)) {
      ok = PyList_Append(found, value) == 0;
      look(value);
      for (Py_ssize_t i = 0; ok && PyList_Check(value) && i < PyList_GET_SIZE(value); ++i) {
        ok = PyList_Append(found, PyList_GET_ITEM(value, i)) == 0;
        look(PyList_GET_ITEM(value, i));
      }
    }
    Py_XDECREF(dict);
    if (!ok) Py_CLEAR(found);
  }
  return found;
}

// sources_new(tensors) -> capsule: their addresses, sizes and versions, their memory held with it
PyObject* py_sources_new(PyObject*, PyObject* const* a, Py_ssize_t n) {
  std::vector<const at::Tensor*> ts;
  if (n != 1 || !list_sources(a[0], &ts)) {
    PyErr_SetString(PyExc_TypeError, "sources_new takes a list of tensors");
    return nullptr;
  }
  std::unique_ptr<std::vector<Source>> made(new std::vector<Source>());
  for (const at::Tensor* t : ts) made->emplace_back(*t);
  PyObject* cap = PyCapsule_New(made.get(), "eagle.sources", [](PyObject* c) {
    delete static_cast<std::vector<Source>*>(PyCapsule_GetPointer(c, "eagle.sources"));
  });
  if (cap) made.release();
  return cap;
}

// sources_current(capsule, tensors): these tensors lie where those lay, and no write to them was counted
PyObject* py_sources_current(PyObject*, PyObject* const* a, Py_ssize_t n) {
  auto* of = n == 2 ? static_cast<std::vector<Source>*>(PyCapsule_GetPointer(a[0], "eagle.sources")) : nullptr;
  std::vector<const at::Tensor*> ts;
  if (!of || !list_sources(a[1], &ts)) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "sources_current takes a capsule and a list of tensors");
    return nullptr;
  }
  if (ts.size() != of->size()) Py_RETURN_FALSE;
  for (size_t i = 0; i < ts.size(); ++i)
    if (!(*of)[i].same(*ts[i])) Py_RETURN_FALSE;
  Py_RETURN_TRUE;
}

// decoder_new(ints, floats, emb, head, norm, inv_freqs, layers, layer_list, cache_type) -> capsule
//   ints: (D, I, H, G, hd, V, form); floats: (eps, rope_factor, scale); layers: per layer (seven projections, qkv, gu,
//   two norms)
PyObject* py_decoder_new(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int v[7];
  float f[3];
  if (n != 9 || !PyArg_ParseTuple(a[0], "iiiiiii", v, v + 1, v + 2, v + 3, v + 4, v + 5, v + 6) ||
      !PyArg_ParseTuple(a[1], "fff", f, f + 1, f + 2) || !PyList_Check(a[6]) || !PyList_Check(a[7])) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "decoder_new takes nine arguments");
    return nullptr;
  }
  std::unique_ptr<Decoder> d(new Decoder());
  d->kept.reserve(PyList_GET_SIZE(a[6]) * 40 + 16);
  d->D = v[0]; d->I = v[1]; d->H = v[2]; d->G = v[3]; d->hd = v[4]; d->V = v[5]; d->form = v[6];
  d->eps = f[0]; d->rope_factor = f[1]; d->scale = f[2];
  d->emb = take_mat(d.get(), a[2]);
  d->head = take_mat(d.get(), a[3]);
  d->norm = take(d.get(), a[4]).data_ptr();
  const Py_ssize_t nl = PyList_GET_SIZE(a[6]);
  d->layers.resize(nl);
  for (Py_ssize_t i = 0; i < nl; ++i) {
    PyObject* t = PyList_GET_ITEM(a[6], i);
    if (!PyTuple_Check(t) || PyTuple_GET_SIZE(t) != NPROJ + 4) throw Bad();
    Layer& l = d->layers[i];
    for (int j = 0; j < NPROJ; ++j) l.p[j] = take_mat(d.get(), PyTuple_GET_ITEM(t, j));
    l.norm1 = take(d.get(), PyTuple_GET_ITEM(t, NPROJ + 2)).data_ptr();
    l.norm2 = take(d.get(), PyTuple_GET_ITEM(t, NPROJ + 3)).data_ptr();
  }
  d->inv_freqs = static_cast<const float*>(take(d.get(), a[5]).data_ptr());
  for (Py_ssize_t i = 0; i < nl; ++i) {
    PyObject* t = PyList_GET_ITEM(a[6], i);
    Layer& l = d->layers[i];
    l.qkv = take_mat(d.get(), PyTuple_GET_ITEM(t, NPROJ));
    l.gu = take_mat(d.get(), PyTuple_GET_ITEM(t, NPROJ + 1));
    d->linear_bias |= l.p[O].bias || l.p[DOWN].bias;
  }
  Py_INCREF(d->layer_list = a[7]);
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(a[7]); ++i) {
    PyObject* o = PyList_GET_ITEM(a[7], i);
    Py_INCREF(o);
    d->layer_items.push_back(o);
  }
  Py_INCREF(d->cache_type = a[8]);
  PyObject* cap = PyCapsule_New(d.get(), "eagle.decoder", destroy);
  if (cap) d.release();
  return cap;
}

// decoder_current(capsule): the layers are the ones the decoder was built from, their tensors lie where they lay, and no
// write to them was counted
PyObject* py_decoder_current(PyObject*, PyObject* const* a, Py_ssize_t n) {
  Decoder* d = n == 1 ? static_cast<Decoder*>(PyCapsule_GetPointer(a[0], "eagle.decoder")) : nullptr;
  if (!d) return nullptr;
  if (PyList_GET_SIZE(d->layer_list) != (Py_ssize_t)d->layer_items.size()) Py_RETURN_FALSE;
  for (size_t i = 0; i < d->layer_items.size(); ++i)
    if (PyList_GET_ITEM(d->layer_list, i) != d->layer_items[i]) Py_RETURN_FALSE;
  for (const Source& s : d->kept)
    if (!s.same()) Py_RETURN_FALSE;
  Py_RETURN_TRUE;
}

// decoder_forward(capsule, ids, caches, mask, Tk, positions, pos_add, pos_step)
//   mask: additive tensor [.., T, Tk] over the last Tk rows, or with Tk = 0 [.., T, S] (its last min(S, 64) columns are
//   read), or None: causal.  positions: int tensor [T] or None, plus pos_add + pos_step * row.
//   Returns the logits [1, T, V] and advances the caches' offsets; None, nothing done, where the arguments are not what
//   this path takes.
PyObject* py_decoder_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  static PyObject *s_keys = str("keys"), *s_values = str("values"), *s_offset = str("_offset");
  Decoder* d = n == 8 ? static_cast<Decoder*>(PyCapsule_GetPointer(a[0], "eagle.decoder")) : nullptr;
  if (!d) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "decoder_forward takes eight arguments");
    return nullptr;
  }
  const at::Tensor *ids = tensor(a[1]), *mask = tensor(a[3]), *pos = tensor(a[5]);
  if (!ids || !ids->is_cuda() || !ids->is_contiguous() || ids->dim() != 2 || ids->size(0) != 1 || ids->size(1) < 1 ||
      (ids->scalar_type() != at::kInt && ids->scalar_type() != at::kLong) || ids->device() != d->kept[0].tensor.device())
    Py_RETURN_NONE;
  const int64_t T = ids->size(1);
  if (T > (a[3] == Py_None ? EAGLE_MAX_CHUNK : EAGLE_MAX_TREE_SLOTS) || (a[3] != Py_None && !mask)) Py_RETURN_NONE;
  if (a[5] != Py_None &&
      !(pos && pos->is_cuda() && pos->is_contiguous() && pos->numel() == T && (pos->scalar_type() == at::kInt || pos->scalar_type() == at::kLong)))
    Py_RETURN_NONE;
  long Tk = PyLong_AsLong(a[4]);
  const long pos_add = PyLong_AsLong(a[6]), pos_step = PyLong_AsLong(a[7]);
  if (PyErr_Occurred()) return nullptr;

  // the caches: of this framework's class, all at one length
  if (!PyList_Check(a[2]) || PyList_GET_SIZE(a[2]) != (Py_ssize_t)d->layers.size() || d->layers.empty()) Py_RETURN_NONE;
  const bool chunk = T > 2 * EAGLE_MAX_TREE;
  const int R = chunk ? (int)((T + 31) / 32 * 32) : (int)T;
  Pass ps{*d, *ids};
  long offset = -1;
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(a[2]); ++i) {
    PyObject* c = PyList_GET_ITEM(a[2], i);
    if ((PyObject*)Py_TYPE(c) != d->cache_type) Py_RETURN_NONE;
    PyObject* attr[3] = {PyObject_GetAttr(c, s_keys), PyObject_GetAttr(c, s_values), PyObject_GetAttr(c, s_offset)};
    bool ok = attr[0] && attr[1] && attr[2] && PyLong_Check(attr[2]);
    if (ok) {
      const long off = PyLong_AsLong(attr[2]);
      const at::Tensor *kt = tensor(attr[0]), *vt = tensor(attr[1]);
      ok = plain(kt, at::kHalf) && plain(vt, at::kHalf) && kt->dim() == 4 && kt->size(0) == 1 && kt->size(1) == d->G &&
           kt->size(3) == d->hd && kt->sizes() == vt->sizes() && (i == 0 || (off == offset && kt->size(2) == ps.cap));
      if (ok) {
        offset = off;
        ps.cap = kt->size(2);
        ps.keys.push_back(kt->data_ptr());
        ps.values.push_back(vt->data_ptr());
      }
    }
    for (PyObject* o : attr) Py_XDECREF(o);
    PyErr_Clear();
    if (!ok) Py_RETURN_NONE;
  }
  const long S = offset + T;
  if (offset < 0 || offset + R > ps.cap) Py_RETURN_NONE;

  eagle_pass_begin b = {};
  if (mask) {
    const int64_t cols = Tk > 0 ? Tk : S;
    if (Tk <= 0) Tk = S < 64 ? S : 64;
    const at::ScalarType mt = mask->scalar_type();
    const int dims = (int)mask->dim();
    if (!mask->is_cuda() || dims < 2 || mask->size(-1) != cols || mask->size(-2) != T || mask->numel() != cols * T ||
        mask->stride(-1) != 1 || Tk > 64 || Tk > S || (mt != at::kHalf && mt != at::kBFloat16 && mt != at::kFloat))
      Py_RETURN_NONE;
    b.mask_bits = mt == at::kFloat ? 32 : 16;
    b.mask_ld = mask->stride(-2);
    b.mask = static_cast<const char*>(mask->data_ptr()) + (cols - Tk) * (b.mask_bits / 8);
  } else {
    Tk = chunk ? 32 : (S < 64 ? S : 64);
  }
  ps.st = stream_of(*ids);
  ps.T = (int)T;
  ps.R = R;
  ps.Tk = (int)Tk;
  ps.S = (int)(chunk ? offset + R : S);
  ps.plan();
  if (chunk && (ps.S < 32 || d->D > 8192)) Py_RETURN_NONE;
  const at::Tensor buffers = empty({(int64_t)ps.ar.size}, at::kByte, *ids);
  ps.ar.base = static_cast<char*>(buffers.data_ptr());
  at::Tensor logits = empty({1, T, d->V}, at::kHalf, *ids);

  b.ids = ids->data_ptr();
  b.ids64 = ids->scalar_type() == at::kLong;
  b.wq = d->emb.w;
  b.scales = d->emb.s;
  b.biases = d->emb.b;
  b.norm_w = d->layers[0].norm1;
  b.eps = d->eps;
  b.h = ps.p(ps.h);
  b.hn = ps.folded ? nullptr : ps.p(ps.hn);
  if (pos) {
    b.positions = pos->data_ptr();
    b.pos64 = pos->scalar_type() == at::kLong;
  }
  b.inv_freqs = d->inv_freqs;
  b.scaling_factor = d->rope_factor;
  b.positions_out = static_cast<int32_t*>(ps.p(ps.pos));
  b.rope_cs = static_cast<float*>(ps.p(ps.cs));
  b.lens = ps.len(0);
  b.T = (int)T;
  b.R = R;
  b.D = d->D;
  b.V = d->emb.N;
  b.half = d->hd / 2;
  b.Tk = (int)Tk;
  b.pos_add = (int)pos_add;
  b.pos_step = (int)pos_step;
  b.write_len = (int)offset;
  b.attn_len = (int)(S - Tk);
  if (chunk)
    b.piece_len = static_cast<int32_t*>(ps.p(ps.pieces));
  else
    b.words = static_cast<uint32_t*>(ps.p(ps.words));
  int rc = eagle_pass_begin_f16(&b, ps.st);
  const int nl = (int)d->layers.size();
  for (int i = 0; rc == EAGLE_OK && i < nl; ++i) rc = ps.layer(i, i + 1 < nl ? d->layers[i + 1].norm1 : d->norm);
  if (rc == EAGLE_OK && ps.folded)
    rc = eagle_rmsnorm_f16(ps.p(ps.h), nullptr, d->norm, d->eps, nullptr, ps.p(ps.hn), (int)T, d->D, ps.st);
  if (rc == EAGLE_OK) rc = ps.product(d->head, ps.p(ps.hn), logits.data_ptr(), (int)T);
  if (rc != EAGLE_OK) return fail(rc, "decoder pass");
  PyObject* end = PyLong_FromLong(S);
  for (Py_ssize_t i = 0; end && i < PyList_GET_SIZE(a[2]); ++i)
    if (PyObject_SetAttr(PyList_GET_ITEM(a[2], i), s_offset, end) < 0) {
      Py_DECREF(end);
      return nullptr;
    }
  Py_XDECREF(end);
  return THPVariable_Wrap(std::move(logits));
}

}  // namespace eagle_host
