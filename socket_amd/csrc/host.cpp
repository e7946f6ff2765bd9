// Host side of calls that are shorter than their own preparation: operands are looked at and handed to the library in
// one step from Python, without a Python object or a ctypes conversion per property.
//
// An append of 2 x 777 rows x 8 heads of 64 is 6.1 us on the GPU; looking its operands over in Python took 3.4 us and the
// call through ctypes 5.1, so a stream of such appends was bound by the host, 10.2 us each: now 5.9, the GPU's own pace, with
// 4.6 of the host's under it.
#include <Python.h>

#include <torch/csrc/autograd/python_variable.h>

#include <exception>

#include "../../include/socket_hip.h"

namespace {

constexpr int kHashDim = 128;      // coordinates the hashing kernel contracts over
PyObject *tensor_type, *parameter_type;

// Exactly a tensor or a parameter: a tracer's or a mode's stand-in for one is neither.
bool plain(PyObject* o) { return (PyObject*)Py_TYPE(o) == tensor_type || (PyObject*)Py_TYPE(o) == parameter_type; }

// An append's operands as the library takes them.
struct Append {
  const void *k, *v, *words;
  void *k_cache, *v_cache, *codes, *v_norm, *lens;
  int64_t k_strides[3], v_strides[3], cache_strides[3];      // of batch, head and row
  int dtype, B, H, S, D;
};

// Whether one call of socket_cache_append takes the rows t[0], t[1] [B,S,H,D] into the cache t[2..6] with planes t[7].
bool fits(const at::Tensor* const* t, Append& a) {
  const at::Tensor &k = *t[0], &v = *t[1], &kc = *t[2], &words = *t[7];
  const at::ScalarType type = kc.scalar_type();
  a.dtype = type == at::kFloat ? SOCKET_F32 : type == at::kBFloat16 ? SOCKET_BF16 : SOCKET_F16;
  if (type != at::kFloat && type != at::kBFloat16 && type != at::kHalf) return false;
  for (int i = 0; i < 8; ++i)
    if (!t[i]->is_cuda() || t[i]->device() != k.device() || (i < 4 && t[i]->scalar_type() != type)) return false;
  if (k.dim() != 4 || kc.dim() != 4 || words.dim() < 2 || k.sizes() != v.sizes()) return false;
  const int64_t B = k.size(0), S = k.size(1), H = k.size(2), D = k.size(3);
  if (H != kc.size(1) || D != kc.size(3) || S < 1 || D % 8 != 0 || D > kHashDim || words.size(1) != kHashDim ||
      kc.size(0) * kc.size(1) > 65535)
    return false;
  for (int i = 2; i < 8; ++i)
    if (!t[i]->is_contiguous()) return false;
  const int order[3] = {0, 2, 1};
  const int64_t piece = 16 / (int64_t)kc.element_size();      // (whole 16-byte pieces throughout)
  if (k.stride(3) != 1 || v.stride(3) != 1) return false;
  for (int i = 0; i < 3; ++i) {
    a.k_strides[i] = k.stride(order[i]);
    a.v_strides[i] = v.stride(order[i]);
    a.cache_strides[i] = kc.stride(i);
    if (a.k_strides[i] % piece != 0 || a.v_strides[i] % piece != 0) return false;
  }
  a.k = k.data_ptr();
  a.v = v.data_ptr();
  a.k_cache = kc.data_ptr();
  a.v_cache = t[3]->data_ptr();
  if (((uintptr_t)a.k | (uintptr_t)a.v | (uintptr_t)a.k_cache | (uintptr_t)a.v_cache) % 16 != 0) return false;
  a.codes = t[4]->data_ptr();
  a.v_norm = t[5]->data_ptr();
  a.lens = t[6]->data_ptr();
  a.words = words.data_ptr();
  a.B = (int)B;
  a.H = (int)H;
  a.S = (int)S;
  a.D = (int)D;
  return true;
}

// cache_append(k, v, k_cache, v_cache, codes, v_norm, lens, words, pos0, L, P, Tcap, stream, run): -1 if the operands do
// not fit, else 0 or, with `run`, the call's status.
PyObject* cache_append(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 14) {
    PyErr_SetString(PyExc_TypeError, "cache_append takes 14 arguments");
    return nullptr;
  }
  long long num[6];      // pos0, L, P, Tcap, stream, run
  for (int i = 0; i < 6; ++i) {
    num[i] = PyLong_AsLongLong(args[8 + i]);
    if (num[i] == -1 && PyErr_Occurred()) return nullptr;
  }
  const at::Tensor* t[8];
  for (int i = 0; i < 8; ++i) {
    if (!plain(args[i])) return PyLong_FromLong(-1);
    t[i] = &THPVariable_Unpack(args[i]);
  }
  Append a;
  try {
    if (!fits(t, a)) return PyLong_FromLong(-1);
  } catch (const std::exception& e) {      // (a sparse tensor has no strides, say)
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
  int status = 0;
  if (num[5]) {
    Py_BEGIN_ALLOW_THREADS
    status = socket_cache_append(a.k, a.v, a.dtype, a.k_strides[0], a.k_strides[1], a.k_strides[2], a.v_strides[0],
                                 a.v_strides[1], a.v_strides[2], a.words, a.k_cache, a.v_cache, a.cache_strides[0],
                                 a.cache_strides[1], a.cache_strides[2], (uint32_t*)a.codes, (uint16_t*)a.v_norm,
                                 (int32_t*)a.lens, (int)num[0], a.B, a.H, a.S, a.D, (int)num[1], (int)num[2], num[3],
                                 (void*)num[4]);
    Py_END_ALLOW_THREADS
  }
  return PyLong_FromLong(status);
}

PyMethodDef methods[] = {
    {"cache_append", (PyCFunction)(void (*)())cache_append, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
  PyObject* torch = PyImport_ImportModule("torch");
  PyObject* nn = torch ? PyImport_ImportModule("torch.nn") : nullptr;
  if (!nn) return nullptr;
  tensor_type = PyObject_GetAttrString(torch, "Tensor");
  parameter_type = PyObject_GetAttrString(nn, "Parameter");
  Py_DECREF(nn);
  Py_DECREF(torch);
  if (!tensor_type || !parameter_type) return nullptr;
  return PyModule_Create(&module);
}
