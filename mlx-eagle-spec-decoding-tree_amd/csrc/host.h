// Shared by the native host path (host.cpp, decoder.cpp): torch tensors in, C-ABI calls out.
#pragma once
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include "../../include/eagle_mi355x.h"

namespace eagle_host {

struct Slot {
  void* ptr = nullptr;
  size_t bytes = 0;
};

inline void* stream_of(const at::Tensor& t) {
  return static_cast<void*>(c10::hip::getCurrentHIPStream(t.device().index()).stream());
}

// nullptr where the object is not a tensor
inline const at::Tensor* tensor(PyObject* o) {
  return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr;
}
inline bool plain(const at::Tensor* t, at::ScalarType dt) {
  return t && t->is_cuda() && t->scalar_type() == dt && t->is_contiguous();
}
inline bool packed(const at::Tensor* t) {
  return t && t->is_cuda() && t->is_contiguous() && t->dim() == 2 &&
         (t->scalar_type() == at::kInt || t->scalar_type() == at::kUInt32);
}
inline at::Tensor empty(at::IntArrayRef sizes, at::ScalarType dt, const at::Tensor& like) {
  return at::empty(sizes, like.options().dtype(dt));
}

// raises what _lib.check raises
PyObject* fail(int rc, const char* what);

// The split-K workspace of the streaming matmul on the device of `like` (ops.workspace keeps it: zeroed
// counters that every call leaves zero, never released once a captured graph may hold its address).
// False with a Python error set.
bool qmm_workspace(const at::Tensor& like, size_t need, Slot* out);

// Whether the operands have the alignment that the small-row kernel asks for
bool small_aligned(const void* x, const void* s, const void* b, const void* bias, const void* out);

// The product on eagle_qmm_rows_w4g64_f16, and whether it is the form to take for up to 64 rows
bool rows_takes(int M, int N, int K, const void* x, const void* s, const void* b, const void* out);
int rows(const at::Tensor& like, const void* x, const void* w, const void* s, const void* b, const void* bias, void* out, int M,
         int N, int K, bool swiglu, void* st);

// The product of M rows: which form runs is the rule of ops.quantized_matmul (its docstring).  A negative
// result: a Python error is set.
int matmul(const at::Tensor& like, const void* x, const void* w, const void* s, const void* b, const void* bias, void* out,
           int M, int N, int K, void* st);

// silu(g) * u of interleaved gate|up rows: the rule of ops.quantized_matmul_swiglu, or with `exact` the one of the native
// decoder, which leaves out the forms that round the weights (the slab kernel for 33..64 rows, the GEMM above)
int swiglu(const at::Tensor& like, const void* x, const void* w, const void* s, const void* b, const void* bias, void* out,
           int M, int N, int K, bool exact, void* st);

PyObject* py_module_parts(PyObject*, PyObject* const* a, Py_ssize_t n);
PyObject* py_sources_new(PyObject*, PyObject* const* a, Py_ssize_t n);
PyObject* py_sources_current(PyObject*, PyObject* const* a, Py_ssize_t n);
PyObject* py_decoder_new(PyObject*, PyObject* const* a, Py_ssize_t n);
PyObject* py_decoder_current(PyObject*, PyObject* const* a, Py_ssize_t n);
PyObject* py_decoder_forward(PyObject*, PyObject* const* a, Py_ssize_t n);

}  // namespace eagle_host
