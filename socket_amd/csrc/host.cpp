// Host side of calls that are shorter than their own preparation: operands are looked at and handed to the library in
// one step from Python, without a Python object or a ctypes conversion per property.
//
// An append of 2 x 777 rows x 8 heads of 64 is 6.1 us on the GPU; looking its operands over in Python took 3.4 us and the
// call through ctypes 5.1, so a stream of such appends was bound by the host, 10.2 us each: now 5.9, the GPU's own pace, with
// 4.6 of the host's under it.
#include <Python.h>

#include <ATen/ops/empty.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
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

// ---- the list builder and the attention over its list -------------------------------------------
//
// Over 4448 tokens of 32 heads (32 tables x 256) the two are some 20 us on the GPU, and their Python took the host 37.5: looking
// operands over, five allocations and four calls through ctypes.  Now 18 to 21, and such a stream of calls 38.5 / 20.5 to 22 us each.
// Operands in another form than these take go the way through Python, which also says what is wrong with them.
int type_of(at::ScalarType t) {
  return t == at::kFloat ? SOCKET_F32 : t == at::kBFloat16 ? SOCKET_BF16 : t == at::kHalf ? SOCKET_F16 : -1;
}

// The first n arguments as tensors of one HIP device.
template <int N>
bool tensors(PyObject* const* args, const at::Tensor* (&t)[N]) {
  for (int i = 0; i < N; ++i) {
    if (!plain(args[i])) return false;
    t[i] = &THPVariable_Unpack(args[i]);
    if (!t[i]->is_cuda() || t[i]->device() != t[0]->device() || t[i]->layout() != at::kStrided) return false;
  }
  return true;
}

PyObject* none() { Py_RETURN_NONE; }

// What a call that did not return 0 is answered with: its name and its status.
PyObject* failed(const char* name, int status) { return Py_BuildValue("si", name, status); }

// build_list(q_probs, k_hard, v_norm, allowed, sink, window, M, max_base, max_M, workspace, stream): (list, lengths), None if
// the operands do not fit, (name, status) of a call that failed.  workspace(device, bytes, zero bytes) is asked where one is needed.
PyObject* build_list(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 11) {
    PyErr_SetString(PyExc_TypeError, "build_list takes 11 arguments");
    return nullptr;
  }
  const at::Tensor* t[4];
  if (!tensors(args, t)) return none();
  long long num[6];      // sink, window, M, max_base, max_M, stream
  for (int i = 0; i < 6; ++i) {
    PyObject* o = args[i < 5 ? 4 + i : 10];
    if (!PyLong_CheckExact(o)) return none();
    num[i] = PyLong_AsLongLong(o);
    if (num[i] == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      return none();
    }
  }
  const at::Tensor &q = *t[0], &k = *t[1], &norms = *t[2], &allowed = *t[3];
  if (q.dim() != 4 || k.dim() != 4 || norms.dim() != 3 || allowed.dim() != 3) return none();
  const int64_t B = q.size(0), H = q.size(1), L = q.size(2), R = q.size(3), T = k.size(3);
  const int64_t M = std::min<int64_t>(num[2], T), rows[3] = {B, H, T};
  if (std::min({B, H, L, R, T, M}) < 1 || B * H > 65535 || std::max({L, R, T}) > INT32_MAX || M > num[4] || k.size(0) != B ||
      k.size(1) != H || k.size(2) != L || norms.sizes() != at::IntArrayRef(rows) || allowed.sizes() != at::IntArrayRef(rows) ||
      k.scalar_type() != at::kShort || allowed.scalar_type() != at::kBool || type_of(q.scalar_type()) < 0 ||
      type_of(norms.scalar_type()) < 0)
    return none();
  for (const at::Tensor* x : t)
    if (!x->is_contiguous()) return none();
  const int64_t sink = std::clamp<int64_t>(num[0], 0, T), window = std::clamp<int64_t>(num[1], 0, T);
  const int64_t base = std::max<int64_t>(1, sink + (window > 0 ? T - std::max(T - window, sink) : 0)), width = base + M;
  if (base > num[3]) return none();
  const size_t bytes = socket_select_workspace_bytes((int)B, (int)H, (int)T, (int)M);
  at::Tensor ws;
  if (bytes > 0) {
    PyObject* device = PyObject_GetAttrString(args[0], "device");
    if (!device) return nullptr;
    PyObject* got = PyObject_CallFunction(args[9], "OKK", device, (unsigned long long)bytes,
                                          (unsigned long long)socket_select_workspace_zero_bytes((int)B, (int)H, (int)T, (int)M));
    Py_DECREF(device);
    if (!got) return nullptr;
    if (THPVariable_Check(got)) ws = THPVariable_Unpack(got);
    Py_DECREF(got);
    if (!ws.defined()) return none();
  }
  const auto on = at::TensorOptions().device(q.device());
  at::Tensor scores = at::empty({B, H, T}, on.dtype(at::kFloat)), list = at::empty({B, H, width}, on.dtype(at::kInt)),
             lengths = at::empty({B, H}, on.dtype(at::kInt));
  const void *pq = q.data_ptr(), *pk = k.data_ptr(), *pn = norms.data_ptr(), *pa = allowed.data_ptr();
  void *ps = scores.data_ptr(), *pl = list.data_ptr(), *pc = lengths.data_ptr(), *pw = bytes > 0 ? ws.data_ptr() : nullptr;
  const int q_type = type_of(q.scalar_type()), norm_type = type_of(norms.scalar_type());
  int scored = 0, selected = 0;
  Py_BEGIN_ALLOW_THREADS
  scored = socket_soft_hash_collision_typed(pq, q_type, (const int16_t*)pk, (const uint8_t*)pa, pn, norm_type, (float*)ps, (int)B, (int)H,
                                            (int)L, (int)R, (int)T, (void*)num[5]);
  if (scored == SOCKET_OK)
    selected = socket_select_list_allowed((const float*)ps, T, (const uint8_t*)pa, (int)B, (int)H, (int)T, (int)M, (int)sink, (int)window,
                                          (int32_t*)pl, width, (int)width, (int32_t*)pc, pw, bytes, (void*)num[5]);
  Py_END_ALLOW_THREADS
  if (scored != SOCKET_OK) return failed("socket_soft_hash_collision", scored);
  if (selected != SOCKET_OK) return failed("socket_select_list", selected);
  PyObject* out[2] = {THPVariable_Wrap(std::move(list)), THPVariable_Wrap(std::move(lengths))};
  PyObject* both = out[0] && out[1] ? PyTuple_Pack(2, out[0], out[1]) : nullptr;
  Py_XDECREF(out[0]);
  Py_XDECREF(out[1]);
  return both;
  END_HANDLE_TH_ERRORS
}

// sparse_attention(query, key, value, list, lengths, stream): the output, None if the operands do not fit, (name, status) of
// a call that failed.
PyObject* sparse_attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6) {
    PyErr_SetString(PyExc_TypeError, "sparse_attention takes 6 arguments");
    return nullptr;
  }
  const at::Tensor* t[5];
  if (!tensors(args, t)) return none();
  const long long stream = PyLong_AsLongLong(args[5]);
  if (stream == -1 && PyErr_Occurred()) return nullptr;
  const at::Tensor &q = *t[0], &k = *t[1], &v = *t[2], &list = *t[3], &lengths = *t[4];
  if (q.dim() != 3 || k.dim() != 4 || v.dim() != 4 || list.dim() != 3 || lengths.dim() != 2) return none();
  const int64_t B = q.size(0), H = q.size(1), D = q.size(2), Hkv = k.size(1), rows = k.size(2), width = list.size(2);
  const int type = type_of(q.scalar_type());
  if (type < 0 || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type() || (D != 16 && D != 32 && D != 64 && D != 128) ||
      k.size(3) != D || v.size(3) != D || q.stride(2) != 1 || k.stride(3) != 1 || v.stride(3) != 1 || std::min({B, H, Hkv, rows, width}) < 1 ||
      H % Hkv != 0 || std::max({B, H, rows, width}) > INT32_MAX || list.scalar_type() != at::kInt || lengths.scalar_type() != at::kInt ||
      list.stride(2) != 1 || k.size(0) != B || v.sizes() != k.sizes() || list.size(0) != B || list.size(1) != H ||
      lengths.sizes() != list.sizes().slice(0, 2))
    return none();
  const size_t bytes = socket_sparse_attention_workspace_bytes((int)B, (int)H, (int)D, (int)width);
  at::Tensor out = at::empty({B, H, D}, at::TensorOptions().device(q.device()).dtype(q.scalar_type())),
             ws = at::empty({(int64_t)(bytes / 4)}, at::TensorOptions().device(q.device()).dtype(at::kFloat));
  const void *pq = q.data_ptr(), *pk = k.data_ptr(), *pv = v.data_ptr(), *pl = list.data_ptr(), *pc = lengths.data_ptr();
  void *po = out.data_ptr(), *pw = ws.data_ptr();
  const int64_t s[10] = {q.stride(0), q.stride(1), k.stride(0), k.stride(1), k.stride(2), v.stride(0), v.stride(1), v.stride(2),
                         list.stride(0), list.stride(1)};
  const int64_t c0 = lengths.stride(0), c1 = lengths.stride(1);
  int status = 0;
  Py_BEGIN_ALLOW_THREADS
  status = socket_sparse_attention(pq, pk, pv, type, s[0], s[1], s[2], s[3], s[4], s[5], s[6], s[7], (const int32_t*)pl, s[8], s[9],
                                   (const int32_t*)pc, c0, c1, po, H * D, D, pw, bytes, (int)B, (int)H, (int)Hkv, (int)D, (int)rows,
                                   (int)width, (void*)stream);
  Py_END_ALLOW_THREADS
  if (status != SOCKET_OK) return failed("socket_sparse_attention", status);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"build_list", (PyCFunction)(void (*)())build_list, METH_FASTCALL, nullptr},
    {"sparse_attention", (PyCFunction)(void (*)())sparse_attention, METH_FASTCALL, nullptr},
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
