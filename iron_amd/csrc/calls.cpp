// The checks and the launch of the operators that a program calls one at a time, as one native call: a product of 192 x 64 x 384 took the host
// 5.6 us through Python's checks and ctypes (3 tensors' checks 0.9, their addresses 0.25, the stream's 0.4, the arguments' conversion 0.9, the launch 2.5)
// where the GPU takes 4.0.  What is not the plain case -- another type of tensor or of number, another dtype, strides, element
// count -- is not decided here: the call answers None, and the caller's Python says what is wrong or does it the long way.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <climits>

namespace {

typedef int (*GemmFn)(const void*, const void*, void*, int, int, int, int, int, const int*, const int*, void*);
typedef int64_t (*GemmRoomFn)(int, int, int, int, int);
typedef int (*GemmSharedFn)(const void*, const void*, void*, int, int, int, int, int, void*, void*);
typedef int (*GemvFn)(const void*, const void*, void*, int, int, int, int, const int*, int, int, void*);
typedef int (*MhaFn)(const void*, const void*, const void*, void*, int, int, int, int, int, int, float, int, int, int, int, const int*, const int*, void*);
GemmFn gemm_fn;
GemmRoomFn gemm_room_fn;
GemmSharedFn gemm_shared_fn;
GemvFn gemv_fn;
MhaFn mha_fn;

// A plain integer of 32 bits.
bool number(PyObject* o, int& to) {
  if (!PyLong_Check(o)) return false;
  int overflow = 0;
  const long v = PyLong_AsLongAndOverflow(o, &overflow);
  if (overflow != 0 || v < INT_MIN || v > INT_MAX) return false;
  to = (int)v;
  return true;
}
// A contiguous bf16 tensor on the GPU of exactly `count` elements; its address.
bool plain(PyObject* o, int64_t count, const at::Tensor*& t, void*& address) {
  if (!THPVariable_CheckExact(o)) return false;
  t = &THPVariable_Unpack(o);
  if (!t->is_cuda() || t->scalar_type() != at::kBFloat16 || !t->is_contiguous() || t->numel() != count) return false;
  address = t->data_ptr();
  return true;
}
// The launch may wait for room in the queue: other threads run meanwhile.
template <class Launch>
PyObject* launched(Launch launch) {
  int code;
  Py_BEGIN_ALLOW_THREADS
  code = launch();
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(code);
}
template <class Call>
PyObject* guarded(Call call) {
  try {
    return call();
  } catch (...) {   // (a tensor without storage, say: the long way raises what it raises)
    Py_RETURN_NONE;
  }
}

PyObject* gemm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    int M, N, K, b_col_maj, c_col_maj;
    const at::Tensor* t;
    void *A, *B, *C;
    if (n != 8 || !number(a[3], M) || !number(a[4], N) || !number(a[5], K) || !number(a[6], b_col_maj) || !number(a[7], c_col_maj) ||
        !plain(a[0], (int64_t)M * K, t, A) || !plain(a[1], (int64_t)K * N, t, B) || !plain(a[2], (int64_t)M * N, t, C))
      Py_RETURN_NONE;
    void* stream = c10::hip::getCurrentHIPStream().stream();
    const int64_t room = gemm_room_fn(M, N, K, b_col_maj, c_col_maj);
    if (room > 0) {
      const at::Tensor sums = at::empty({room}, t->options().dtype(at::kByte));
      void* workspace = sums.data_ptr();
      return launched([&] { return gemm_shared_fn(A, B, C, M, N, K, b_col_maj, c_col_maj, workspace, stream); });
    }
    return launched([&] { return gemm_fn(A, B, C, M, N, K, b_col_maj, c_col_maj, nullptr, nullptr, stream); });
  });
}

PyObject* gemv(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    int M, K;
    const at::Tensor* t;
    void *W, *x, *y;
    if (n != 5 || !number(a[3], M) || !number(a[4], K) || !plain(a[0], (int64_t)M * K, t, W) || !plain(a[1], K, t, x) || !plain(a[2], M, t, y))
      Py_RETURN_NONE;
    void* stream = c10::hip::getCurrentHIPStream().stream();
    return launched([&] { return gemv_fn(W, x, y, M, K, 1, 1, nullptr, 0, 0, stream); });
  });
}

PyObject* mha_prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    int v[10];   // heads, kv_heads, d, seq, seq_len, kv_len, causal, window, q_interleaved, kv_interleaved
    if (n != 15 || !PyFloat_CheckExact(a[4])) Py_RETURN_NONE;
    for (int i = 0; i < 10; ++i)
      if (!number(a[5 + i], v[i])) Py_RETURN_NONE;
    const at::Tensor* t;
    void *Q, *K, *V, *O;
    const int64_t q = (int64_t)v[3] * v[0], kv = (int64_t)v[5] * v[1];
    if (q < 0 || q > INT_MAX || kv < 0 || kv > INT_MAX || !plain(a[0], q * v[2], t, Q) || !plain(a[1], kv * v[2], t, K) ||
        !plain(a[2], kv * v[2], t, V) || !plain(a[3], q * v[2], t, O))
      Py_RETURN_NONE;
    const float scale = (float)PyFloat_AS_DOUBLE(a[4]);
    void* stream = c10::hip::getCurrentHIPStream().stream();
    return launched([&] { return mha_fn(Q, K, V, O, v[0], v[1], v[2], v[3], v[4], v[5], scale, v[6], v[7], v[8], v[9], nullptr, nullptr, stream); });
  });
}

// The entry points' addresses, from the library that the other calls go to.
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  void* at[5];
  if (n != 5) {
    PyErr_SetString(PyExc_TypeError, "bind: five addresses");
    return nullptr;
  }
  for (int i = 0; i < 5; ++i) {
    at[i] = PyLong_AsVoidPtr(a[i]);
    if (at[i] == nullptr) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: a null address");
      return nullptr;
    }
  }
  gemm_fn = (GemmFn)at[0];
  gemm_room_fn = (GemmRoomFn)at[1];
  gemm_shared_fn = (GemmSharedFn)at[2];
  gemv_fn = (GemvFn)at[3];
  mha_fn = (MhaFn)at[4];
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, "bind(gemm, gemm_workspace_bytes, gemm_shared, gemv_tuned, mha_prefill): their addresses"},
    {"gemm", (PyCFunction)(void (*)(void))gemm, METH_FASTCALL, "gemm(A, B, C, M, N, K, b_col_maj, c_col_maj) -> code, or None"},
    {"gemv", (PyCFunction)(void (*)(void))gemv, METH_FASTCALL, "gemv(W, x, y, M, K) -> code, or None"},
    {"mha_prefill", (PyCFunction)(void (*)(void))mha_prefill, METH_FASTCALL,
     "mha_prefill(Q, K, V, O, scale, heads, kv_heads, d, seq, seq_len, kv_len, causal, window, q_interleaved, kv_interleaved) -> code, or None"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", "Operators checked and launched in one native call.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls(void) { return PyModule_Create(&module); }
