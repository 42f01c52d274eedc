// The host path of the operators in native code: argument checks, result allocation and launches
// behind one METH_FASTCALL entry each, on torch tensors, through the C ABI of the kernel library.
//
// What bounds a small product on this card is not its kernel (6 us for 3584 x 3584) but the call: the
// same checks and the launch in Python through ctypes took 12 us, longer than the kernel, so a stream of
// calls left the GPU idle half of the time.  Here a call costs about as much as the launch itself.
//
// Every function returns None when an argument is not in the plain form (a device tensor of the expected
// type, contiguous, of matching shape): the Python caller then normalises the arguments, or raises the
// error it always raised, and calls again.
#include "host.h"

using namespace eagle_host;

namespace {
PyObject* g_workspace = nullptr;     // ops.workspace(tag, nbytes, device)
constexpr int MAX_DEVICES = 64;
constexpr int POST_SPINS = 4000;     // about 50 us of pauses
Slot g_qmm_ws[MAX_DEVICES];
}  // namespace

namespace eagle_host {

PyObject* fail(int rc, const char* what) {
  if (rc >= 0)
    PyErr_Format(rc >= EAGLE_ERR_NULL && rc <= EAGLE_ERR_WORKSPACE ? PyExc_ValueError : PyExc_RuntimeError,
                 "%s: %s (status %d)", what, eagle_status_string(rc), rc);
  return nullptr;
}

bool qmm_workspace(const at::Tensor& like, size_t need, Slot* out) {
  const int dev = like.device().index();
  if (dev < 0 || dev >= MAX_DEVICES) {
    PyErr_SetString(PyExc_RuntimeError, "device index out of range");
    return false;
  }
  Slot& s = g_qmm_ws[dev];
  if (s.bytes < need) {
    PyObject* d = THPVariable_Wrap(like);
    PyObject* device = d ? PyObject_GetAttrString(d, "device") : nullptr;
    PyObject* t = device ? PyObject_CallFunction(g_workspace, "snO", "qmm", (Py_ssize_t)need, device) : nullptr;
    Py_XDECREF(d);
    Py_XDECREF(device);
    if (!t) return false;
    const at::Tensor& ws = THPVariable_Unpack(t);
    s.ptr = ws.data_ptr();
    s.bytes = (size_t)ws.numel();
    Py_DECREF(t);
  }
  *out = s;
  return true;
}

// the many-row product, split over K where the library says so
static int gemm(const at::Tensor& like, const void* x, const void* w, const void* s, const void* b, const void* bias, void* out, int M,
                int N, int K, bool swiglu, void* st) {
  // the partial sums go back to torch's allocator with the launches in the stream
  const size_t need = eagle_qmm_gemm_workspace_bytes(M, N, K, swiglu);
  at::Tensor ws;
  if (need) ws = empty({(int64_t)need}, at::kByte, like);
  return eagle_qmm_gemm_split_w4g64_f16(x, static_cast<const uint32_t*>(w), s, b, bias, out, M, N, K, 64, 4, swiglu,
                                        need ? ws.data_ptr() : nullptr, need, st);
}

bool rows_takes(int M, int N, int K, const void* x, const void* s, const void* b, const void* out) {
  return eagle_qmm_rows_preferred(M, N, K) && small_aligned(x, s, b, nullptr, out);
}

int rows(const at::Tensor& like, const void* x, const void* w, const void* s, const void* b, const void* bias, void* out, int M,
         int N, int K, bool swiglu, void* st) {
  // the partial sums go back to torch's allocator with the launches in the stream
  const size_t need = eagle_qmm_rows_workspace_bytes(M, N, K);
  at::Tensor ws;
  if (need) ws = empty({(int64_t)need}, at::kByte, like);
  return eagle_qmm_rows_w4g64_f16(x, static_cast<const uint32_t*>(w), s, b, bias, out, M, N, K, 64, 4, swiglu,
                                  need ? ws.data_ptr() : nullptr, need, st);
}

// what the small-row kernel asks of its operands beyond the other forms
bool small_aligned(const void* x, const void* s, const void* b, const void* bias, const void* out) {
  auto low = [](const void* p, uintptr_t bits) { return reinterpret_cast<uintptr_t>(p) & bits; };
  return !low(x, 15) && !low(out, 15) && !low(s, 3) && !low(b, 3) && !low(bias, 7) && x != out;
}

int matmul(const at::Tensor& like, const void* x, const void* w, const void* s, const void* b, const void* bias, void* out,
           int M, int N, int K, void* st) {
  const uint32_t* wq = static_cast<const uint32_t*>(w);
  if (M > 2 * EAGLE_MAX_M) return gemm(like, x, w, s, b, bias, out, M, N, K, false, st);
  if (M > EAGLE_MAX_M && rows_takes(M, N, K, x, s, b, out)) return rows(like, x, w, s, b, bias, out, M, N, K, false, st);
  for (int r0 = 0; r0 < M; r0 += EAGLE_MAX_M) {
    const int m = M - r0 < EAGLE_MAX_M ? M - r0 : EAGLE_MAX_M;
    const void* xr = static_cast<const char*>(x) + (size_t)r0 * K * 2;
    void* outr = static_cast<char*>(out) + (size_t)r0 * N * 2;
    int rc;
    if (eagle_qmm_small_preferred(m, N, K) && small_aligned(xr, s, b, bias, outr)) {
      rc = eagle_qmm_small_w4g64_f16(xr, nullptr, 0.f, wq, s, b, bias, nullptr, outr, m, N, K, 64, 4, 0, st);
    } else if (eagle_qmv_preferred(m, N, K)) {
      rc = eagle_qmv_rows_w4g64_f16(xr, wq, s, b, bias, outr, m, N, K, 64, 4, st);
    } else if (rows_takes(m, N, K, xr, s, b, outr)) {
      rc = rows(like, xr, w, s, b, bias, outr, m, N, K, false, st);
    } else {
      Slot ws;
      if (!qmm_workspace(like, eagle_qmm_workspace_bytes(m, N, K), &ws)) return -1;
      rc = eagle_qmm_w4g64_f16(xr, wq, s, b, bias, outr, m, N, K, 64, 4, ws.ptr, ws.bytes, st);
    }
    if (rc != EAGLE_OK) return rc;
  }
  return EAGLE_OK;
}

// what the slab kernel's SwiGLU form asks of the scales: whole fetches of eight groups, or of two for a ragged K
static bool slab_aligned(const void* x, const void* s, const void* b, const void* bias, const void* out, int K) {
  auto low = [](const void* p, uintptr_t bits) { return reinterpret_cast<uintptr_t>(p) & bits; };
  const uintptr_t bits = K % 512 ? 3 : 15;
  return !low(x, 15) && !low(out, 15) && !low(s, bits) && !low(b, bits) && !low(bias, 1);
}

int swiglu(const at::Tensor& like, const void* x, const void* w, const void* s, const void* b, const void* bias, void* out,
           int M, int N, int K, bool exact, void* st) {
  const uint32_t* wq = static_cast<const uint32_t*>(w);
  if (M > 2 * EAGLE_MAX_M && !exact) return gemm(like, x, w, s, b, bias, out, M, N, K, true, st);
  if (eagle_qmm_small_preferred(M, N, K) && eagle_qmm_small_supported(M, N, K, 0, 1) && small_aligned(x, s, b, bias, out))
    return eagle_qmm_small_w4g64_f16(x, nullptr, 0.f, wq, s, b, bias, nullptr, out, M, N, K, 64, 4, 1, st);
  if (M > EAGLE_MAX_M && !exact && eagle_qmm_slab_swiglu_preferred(M, N, K) && slab_aligned(x, s, b, bias, out, K))
    return eagle_qmm_slab_swiglu_w4g64_f16(x, wq, s, b, bias, out, M, N, K, 64, 4, st);
  if (N % 32 == 0 && (M > 2 * EAGLE_MAX_M ? eagle_qmm_rows_supported(M, N, K, 1) && small_aligned(x, s, b, nullptr, out)
                                          : rows_takes(M, N, K, x, s, b, out)))
    return rows(like, x, w, s, b, bias, out, M, N, K, true, st);
  for (int r0 = 0; r0 < M; r0 += EAGLE_MAX_M) {
    const int m = M - r0 < EAGLE_MAX_M ? M - r0 : EAGLE_MAX_M;
    Slot ws;
    if (!qmm_workspace(like, eagle_qmm_workspace_bytes(m, N, K), &ws)) return -1;
    const int rc = eagle_qmm_swiglu_w4g64_f16(static_cast<const char*>(x) + (size_t)r0 * K * 2, wq, s, b, bias,
                                              static_cast<char*>(out) + (size_t)r0 * N, m, N, K, 64, 4, ws.ptr, ws.bytes, st);
    if (rc != EAGLE_OK) return rc;
  }
  return EAGLE_OK;
}

}  // namespace eagle_host

namespace {

// (x, w_q, scales, biases, bias, out) of a plain product, or of gate|up with SwiGLU
PyObject* product(PyObject* const* a, Py_ssize_t n, bool swi, const char* name) {
  if (n != 6) {
    PyErr_Format(PyExc_TypeError, "%s takes six arguments", name);
    return nullptr;
  }
  const at::Tensor *x = tensor(a[0]), *w = tensor(a[1]), *s = tensor(a[2]), *b = tensor(a[3]), *bias = tensor(a[4]),
                   *out = tensor(a[5]);
  if (!plain(x, at::kHalf) || !packed(w) || !plain(s, at::kHalf) || !plain(b, at::kHalf) || x->dim() < 1) Py_RETURN_NONE;
  const int64_t K = x->size(-1), N = w->size(0);
  if (K < 1 || w->size(1) * 8 != K || s->dim() != 2 || s->size(0) != N || s->size(1) * 64 != K || b->dim() != 2 ||
      b->size(0) != N || b->size(1) * 64 != K)
    Py_RETURN_NONE;
  if (a[4] != Py_None && !(plain(bias, at::kHalf) && bias->dim() == 1 && bias->size(0) == N)) Py_RETURN_NONE;
  const int64_t M = x->numel() / K;
  if (M < 1 || M > INT32_MAX || N > INT32_MAX || K > INT32_MAX) Py_RETURN_NONE;
  const int64_t cols = swi ? N / 2 : N;
  at::Tensor made;
  if (a[5] == Py_None) {
    at::DimVector sizes(x->sizes());
    sizes.back() = cols;
    made = empty(sizes, at::kHalf, *x);
  } else if (!plain(out, at::kHalf) || (swi ? out->numel() < M * cols : out->numel() != M * cols)) {
    Py_RETURN_NONE;                        // (the SwiGLU form has always taken a buffer with room to spare)
  }
  const at::Tensor& o = a[5] == Py_None ? made : *out;
  const void* bp = bias ? bias->data_ptr() : nullptr;
  void* st = stream_of(*x);
  const int rc = swi ? swiglu(*x, x->data_ptr(), w->data_ptr(), s->data_ptr(), b->data_ptr(), bp, o.data_ptr(), (int)M, (int)N, (int)K,
                              false, st)
                     : matmul(*x, x->data_ptr(), w->data_ptr(), s->data_ptr(), b->data_ptr(), bp, o.data_ptr(), (int)M, (int)N, (int)K,
                              st);
  if (rc != EAGLE_OK) return fail(rc, name);
  if (a[5] == Py_None) return THPVariable_Wrap(std::move(made));
  Py_INCREF(a[5]);
  return a[5];
}

PyObject* py_quantized_matmul(PyObject*, PyObject* const* a, Py_ssize_t n) { return product(a, n, false, "quantized_matmul"); }
PyObject* py_quantized_matmul_swiglu(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return product(a, n, true, "quantized_matmul_swiglu");
}

// rope_kv_append(q_lin, k_lin, v_lin, positions, inv_freqs, scaling_factor, q_out, k_cache, v_cache, len_dev, H, G,
//                hd, row_stride, rope_cs)
PyObject* py_rope_kv_append(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 15) {
    PyErr_SetString(PyExc_TypeError, "rope_kv_append takes fifteen arguments");
    return nullptr;
  }
  const at::Tensor *q = tensor(a[0]), *k = tensor(a[1]), *v = tensor(a[2]), *pos = tensor(a[3]), *inv = tensor(a[4]),
                   *qo = tensor(a[6]), *kc = tensor(a[7]), *vc = tensor(a[8]), *len = tensor(a[9]), *cs = tensor(a[14]);
  if (!q || !q->is_cuda() || !k || !v || !qo || !kc || !vc || !len || kc->dim() < 2 || (!cs && (!pos || !inv))) Py_RETURN_NONE;
  const double f = PyFloat_AsDouble(a[5]);
  const long H = PyLong_AsLong(a[10]), G = PyLong_AsLong(a[11]), hd = PyLong_AsLong(a[12]), rs = PyLong_AsLong(a[13]);
  if (PyErr_Occurred()) return nullptr;
  const int T = (int)q->size(0);
  const long cap = kc->size(1);
  void* st = stream_of(*q);
  int rc;
  if (cs)
    rc = eagle_rope_kv_append_table_f16(q->data_ptr(), k->data_ptr(), v->data_ptr(), static_cast<const float*>(cs->data_ptr()),
                                        qo->data_ptr(), kc->data_ptr(), vc->data_ptr(), static_cast<const int32_t*>(len->data_ptr()),
                                        T, (int)H, (int)G, (int)hd, cap, rs, st);
  else
    rc = eagle_rope_kv_append_f16(q->data_ptr(), k->data_ptr(), v->data_ptr(), static_cast<const int32_t*>(pos->data_ptr()),
                                  static_cast<const float*>(inv->data_ptr()), (float)f, qo->data_ptr(), kc->data_ptr(), vc->data_ptr(),
                                  static_cast<const int32_t*>(len->data_ptr()), T, (int)H, (int)G, (int)hd, cap, rs, st);
  if (rc != EAGLE_OK) return fail(rc, "rope_kv_append");
  Py_RETURN_TRUE;
}

// tree_attention(q, k_cache, v_cache, mask_bits, len_dev, scale, max_len, out): one mask word per token, or two
PyObject* py_tree_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 8) {
    PyErr_SetString(PyExc_TypeError, "tree_attention takes eight arguments");
    return nullptr;
  }
  const at::Tensor *q = tensor(a[0]), *k = tensor(a[1]), *v = tensor(a[2]), *m = tensor(a[3]), *len = tensor(a[4]),
                   *out = tensor(a[7]);
  if (!q || !q->is_cuda() || q->dim() != 3 || !k || !k->is_cuda() || k->dim() != 3 || !v || !v->is_cuda() || !m ||
      !m->is_cuda() || !len || !len->is_cuda())
    Py_RETURN_NONE;
  const int H = (int)q->size(0), T = (int)q->size(1), hd = (int)q->size(2), G = (int)k->size(0);
  const long cap = k->size(1);
  const bool wide = m->dim() == 2;
  if (wide && !(m->size(0) == T && m->size(1) == 2)) Py_RETURN_NONE;
  const double scale = PyFloat_AsDouble(a[5]);
  const long max_len = a[6] == Py_None ? cap : PyLong_AsLong(a[6]);
  if (PyErr_Occurred()) return nullptr;
  if (a[7] != Py_None && !plain(out, at::kHalf)) Py_RETURN_NONE;
  at::Tensor made;
  if (a[7] == Py_None) made = empty({T, (int64_t)H * hd}, at::kHalf, *q);
  const at::Tensor& o = a[7] == Py_None ? made : *out;
  // the key splits' partial results, from torch's allocator and back to it when the launches are in the stream
  const size_t need = wide ? eagle_tree_attention_wide_workspace_bytes(T, H, hd, (int)max_len)
                           : eagle_tree_attention_workspace_bytes(H, hd, (int)max_len);
  const at::Tensor ws = empty({(int64_t)need}, at::kByte, *q);
  void* st = stream_of(*q);
  const uint32_t* bits = static_cast<const uint32_t*>(m->data_ptr());
  const int32_t* len_dev = static_cast<const int32_t*>(len->data_ptr());
  const int rc =
      wide ? eagle_tree_attention_wide_f16(q->data_ptr(), k->data_ptr(), v->data_ptr(), bits, len_dev, o.data_ptr(), T, T, H, G,
                                           hd, cap, (int)max_len, (float)scale, ws.data_ptr(), need, st)
           : eagle_tree_attention_f16(q->data_ptr(), k->data_ptr(), v->data_ptr(), bits, len_dev, o.data_ptr(), T, H, G, hd, cap,
                                      (int)max_len, (float)scale, ws.data_ptr(), need, st);
  if (rc != EAGLE_OK) return fail(rc, "tree_attention");
  if (a[7] == Py_None) return THPVariable_Wrap(std::move(made));
  Py_INCREF(a[7]);
  return a[7];
}

// The tensors of a list as segments (device pointers and element counts); false where one is not plain
struct Segments {
  const void* ptr[EAGLE_MAX_SEGMENTS];
  int count[EAGLE_MAX_SEGMENTS];
  int n = 0, total = 0;
};
bool segments(PyObject* list, at::ScalarType dt, bool batched, Segments* s) {
  PyObject* seq = PySequence_Fast(list, "a list of tensors");
  if (!seq) {
    PyErr_Clear();
    return false;
  }
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
  bool ok = n >= 1 && n <= EAGLE_MAX_SEGMENTS;
  for (Py_ssize_t i = 0; ok && i < n; ++i) {
    const at::Tensor* t = tensor(PySequence_Fast_GET_ITEM(seq, i));
    ok = plain(t, dt) && t->numel() >= 1 && t->numel() <= 4096 && (!batched || (t->dim() >= 1 && t->size(0) == 1));
    if (ok) {
      s->ptr[i] = t->data_ptr();
      s->count[i] = (int)t->numel();
      s->total += (int)t->numel();
    }
  }
  s->n = ok ? (int)n : 0;
  Py_DECREF(seq);
  return ok;
}

// process_draft_tree(scores, tokens, parents, sampled_token, k, total): lists of per-level tensors of batch 1
PyObject* py_process_draft_tree(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 6) {
    PyErr_SetString(PyExc_TypeError, "process_draft_tree takes six arguments");
    return nullptr;
  }
  Segments sc, tk, pa;
  const at::Tensor* root = tensor(a[3]);
  if (!segments(a[0], at::kHalf, true, &sc) || !segments(a[1], at::kInt, true, &tk) ||
      !segments(a[2], at::kInt, false, &pa) ||
      !(root && root->is_cuda() && root->numel() >= 1 && (root->scalar_type() == at::kInt || root->scalar_type() == at::kLong)))
    Py_RETURN_NONE;
  const long k = PyLong_AsLong(a[4]), total = PyLong_AsLong(a[5]);
  if (PyErr_Occurred()) return nullptr;
  if (sc.n != tk.n) Py_RETURN_NONE;
  for (int i = 0; i < sc.n; ++i)
    if (sc.count[i] != tk.count[i]) Py_RETURN_NONE;
  if (k < 1 || sc.total % k != 0 || pa.total < sc.total / k) Py_RETURN_NONE;
  const int64_t T = total + 1;
  at::Tensor pos = empty({T}, at::kInt, *root), idx = empty({(int64_t)total}, at::kInt, *root),
             toks = empty({1, T}, at::kInt, *root), mask = empty({T, T}, at::kBFloat16, *root);
  const int rc = eagle_process_draft_tree_lists(
      sc.ptr, reinterpret_cast<const int32_t* const*>(tk.ptr), sc.count, sc.n,
      reinterpret_cast<const uint32_t* const*>(pa.ptr), pa.count, pa.n, root->data_ptr(), root->scalar_type() == at::kLong, (int)k,
      (int)total, static_cast<int32_t*>(pos.data_ptr()), static_cast<int32_t*>(idx.data_ptr()),
      static_cast<int32_t*>(toks.data_ptr()), mask.data_ptr(), stream_of(*root));
  if (rc != EAGLE_OK) return fail(rc, "process_draft_tree");
  PyObject* r = PyTuple_New(4);
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(std::move(pos)));
  PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(std::move(idx)));
  PyTuple_SET_ITEM(r, 2, THPVariable_Wrap(std::move(toks)));
  PyTuple_SET_ITEM(r, 3, THPVariable_Wrap(std::move(mask)));
  return r;
}

// post_process_draft_tree(tree_position_ids, mask_index, total) -> retrieve_indices [leaves, depth + 1].  The result's
// shape is data, so the host waits for it; the rows are written without padding, so that what the wait
// is for is two numbers, which the kernel puts into pinned host memory with one store.  The host watches that
// word for a while before it waits for the stream: the end of a stream is seen 5 us later than the store (39
// nodes with the layout before it: 25.6 us without watching, 20.0 with).  A word that stays zero (a kernel that waits behind other work, a stream
// in capture, an error) ends in the wait.
PyObject* py_post_process_draft_tree(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 3) {
    PyErr_SetString(PyExc_TypeError, "post_process_draft_tree takes three arguments");
    return nullptr;
  }
  const at::Tensor *pos = tensor(a[0]), *idx = tensor(a[1]);
  const long total = PyLong_AsLong(a[2]);
  if (PyErr_Occurred()) return nullptr;
  if (!plain(pos, at::kInt) || !plain(idx, at::kInt) || pos->numel() != total + 1 || idx->numel() != total) Py_RETURN_NONE;
  const c10::hip::HIPStream st = c10::hip::getCurrentHIPStream(pos->device().index());
  at::Tensor full = empty({EAGLE_MAX_TREE_SLOTS * EAGLE_MAX_TREE_SLOTS}, at::kInt, *pos);
  at::Tensor shape = at::empty({2}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
  volatile uint64_t* word = static_cast<volatile uint64_t*>(shape.data_ptr());
  *word = 0;                               // (there is at least one leaf)
  const int rc = eagle_post_process_draft_tree_packed(
      static_cast<const int32_t*>(pos->data_ptr()), static_cast<const int32_t*>(idx->data_ptr()), (int)total,
      static_cast<int32_t*>(full.data_ptr()), static_cast<int32_t*>(shape.data_ptr()), static_cast<void*>(st.stream()));
  if (rc != EAGLE_OK) return fail(rc, "post_process_draft_tree");
  hipError_t err = hipSuccess;
  Py_BEGIN_ALLOW_THREADS
  for (int i = 0; i < POST_SPINS && *word == 0; ++i) __builtin_ia32_pause();
  if (*word == 0) err = hipStreamSynchronize(st.stream());
  Py_END_ALLOW_THREADS
  if (err != hipSuccess) return fail(EAGLE_ERR_HIP, "post_process_draft_tree");
  const uint64_t seen = *word;
  const int64_t leaves = (int32_t)(uint32_t)seen, cols = (int32_t)(seen >> 32);
  if (leaves < 1 || leaves > EAGLE_MAX_TREE_SLOTS || cols < 1 || cols > EAGLE_MAX_TREE_SLOTS) Py_RETURN_NONE;
  return THPVariable_Wrap(full.narrow(0, 0, leaves * cols).view({leaves, cols}));
}

// tile_parts(weights, scales, biases, interleave, wt, sbt, max_scale): one tiled copy of a list of matrices
// (eagle_qmm_tile_parts_w4g64), max_scale a float32 scalar on the device
PyObject* py_tile_parts(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 7 || !PyList_Check(a[0]) || !PyList_Check(a[1]) || !PyList_Check(a[2])) {
    PyErr_SetString(PyExc_TypeError, "tile_parts takes three lists and four more arguments");
    return nullptr;
  }
  const Py_ssize_t parts = PyList_GET_SIZE(a[0]);
  const at::Tensor *wt = tensor(a[4]), *sbt = tensor(a[5]), *mx = tensor(a[6]);
  if (parts < 1 || parts > EAGLE_MAX_TILE_PARTS || PyList_GET_SIZE(a[1]) != parts || PyList_GET_SIZE(a[2]) != parts ||
      !wt || !wt->is_cuda() || !wt->is_contiguous() || !plain(sbt, at::kHalf) || !plain(mx, at::kFloat))
    Py_RETURN_NONE;
  const uint32_t* w[EAGLE_MAX_TILE_PARTS];
  const void *s[EAGLE_MAX_TILE_PARTS], *b[EAGLE_MAX_TILE_PARTS];
  int rows[EAGLE_MAX_TILE_PARTS];
  int64_t N = 0, K = 0;
  for (Py_ssize_t i = 0; i < parts; ++i) {
    const at::Tensor *wi = tensor(PyList_GET_ITEM(a[0], i)), *si = tensor(PyList_GET_ITEM(a[1], i)),
                     *bi = tensor(PyList_GET_ITEM(a[2], i));
    if (!packed(wi) || !plain(si, at::kHalf) || !plain(bi, at::kHalf)) Py_RETURN_NONE;
    if (i == 0) K = wi->size(1) * 8;
    if (wi->size(1) * 8 != K || si->numel() * 64 != wi->size(0) * K || bi->numel() * 64 != wi->size(0) * K) Py_RETURN_NONE;
    w[i] = static_cast<const uint32_t*>(wi->data_ptr());
    s[i] = si->data_ptr();
    b[i] = bi->data_ptr();
    rows[i] = (int)wi->size(0);
    N += wi->size(0);
  }
  if (wt->numel() * wt->element_size() < N * K / 2 || sbt->numel() < N * (K / 64) * 2) Py_RETURN_NONE;
  const int rc = eagle_qmm_tile_parts_w4g64(w, s, b, rows, (int)parts, PyObject_IsTrue(a[3]), static_cast<uint32_t*>(wt->data_ptr()),
                                            sbt->data_ptr(), (int)N, (int)K, static_cast<unsigned*>(mx->data_ptr()), stream_of(*wt));
  if (rc != EAGLE_OK) return fail(rc, "tile_weights");
  Py_RETURN_TRUE;
}

// init(workspace): ops.workspace, which keeps the buffers that outlive a call
PyObject* py_init(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 1 || !PyCallable_Check(a[0])) {
    PyErr_SetString(PyExc_TypeError, "init takes the workspace function");
    return nullptr;
  }
  Py_INCREF(a[0]);
  Py_XSETREF(g_workspace, a[0]);
  Py_RETURN_NONE;
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  try {
    return F(self, a, n);
  } catch (const std::exception& e) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

#define EAGLE_PY(name) {#name, reinterpret_cast<PyCFunction>(&guarded<py_##name>), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {EAGLE_PY(init),
                         EAGLE_PY(quantized_matmul),
                         EAGLE_PY(quantized_matmul_swiglu),
                         EAGLE_PY(rope_kv_append),
                         EAGLE_PY(tree_attention),
                         EAGLE_PY(process_draft_tree),
                         EAGLE_PY(post_process_draft_tree),
                         EAGLE_PY(tile_parts),
                         EAGLE_PY(module_parts),
                         EAGLE_PY(sources_new),
                         EAGLE_PY(sources_current),
                         EAGLE_PY(decoder_new),
                         EAGLE_PY(decoder_current),
                         EAGLE_PY(decoder_forward),
                         {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&module); }
