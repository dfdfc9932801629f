// The host path of the tensor front end (relax_amd/ops.py, relax_amd/module.py) as a CPython extension: argument
// checks, output allocation and the call into the C ABI without one interpreted step per check.  A decode
// projection runs for 4 - 12 us on the device; the same path in Python with ctypes took 10 - 11 us per call, so a chain
// of them was paced by the host (one token through eight 4096 / 11008 layers: 350 - 380 us per pass where the same
// launches replayed from a graph take 280).
//
// Every function takes exactly what the Python function has been handed and accepts only the ordinary case --
// exact tensors of the expected types, shapes and devices.  Anything else returns None without a side effect,
// and the caller runs its Python path, which reports the error (or serves a case not covered here).
// A return value of False is a call that the C ABI refused: its message is in mi355x_wq_last_error.
// Tensor accessors throw for tensors without plain storage (sparse, nested, batched by a transform): no exception
// leaves an entry, such a call is one not taken here.
//
// The C ABI is reached through addresses the Python side passes to bind() -- those of the library it has loaded --, so
// this file links against nothing of the library.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/mi355x_wq.h"
#include "../../include/mi355x_wq_module.h"

namespace {

struct Abi {
  decltype(&mi355x_wq_matmul_fused_ex) fused_ex = nullptr;
  decltype(&mi355x_wq_matmul_tiled_ex) tiled_ex = nullptr;
  decltype(&mi355x_wq_matmul_ws) ws = nullptr;
  decltype(&mi355x_wq_dequantize) dequantize = nullptr;
} abi;

PyObject* none() { Py_RETURN_NONE; }

bool exact_tensor(PyObject* o) { return THPVariable_CheckExact(o); }

// a device tensor of the given type, compact row-major
bool plain(const at::Tensor& t, at::ScalarType type) { return t.is_cuda() && t.scalar_type() == type && t.is_contiguous(); }

bool packed_words(const at::Tensor& t) {
  return t.is_cuda() && (t.scalar_type() == at::kInt || t.scalar_type() == at::kUInt32) && t.is_contiguous() && t.dim() == 2;
}

bool take_int(PyObject* o, int64_t* out) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  *out = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}

// the stream argument of the front end: None (torch's current stream) or an object with a `cuda_stream` handle
bool take_stream(PyObject* o, void** out) {
  if (o == Py_None) {
    *out = c10::hip::getCurrentHIPStream().stream();
    return true;
  }
  PyObject* h = PyObject_GetAttrString(o, "cuda_stream");
  if (h == nullptr) {
    PyErr_Clear();
    return false;
  }
  *out = PyLong_AsVoidPtr(h);
  Py_DECREF(h);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

PyObject* bind(PyObject*, PyObject* args) {
  unsigned long long a, b, c, d;
  if (!PyArg_ParseTuple(args, "KKKK", &a, &b, &c, &d)) return nullptr;
  abi.fused_ex = reinterpret_cast<decltype(abi.fused_ex)>(a);
  abi.tiled_ex = reinterpret_cast<decltype(abi.tiled_ex)>(b);
  abi.ws = reinterpret_cast<decltype(abi.ws)>(c);
  abi.dequantize = reinterpret_cast<decltype(abi.dequantize)>(d);
  Py_RETURN_NONE;
}

// matmul(x, wq, scales, bits, group, zero_point, out, kernel, stream, bias, activation, residual, tiled_n, workspace):
// `kernel` carries the variant in its upper bits, `activation` is MI355X_WQ_ACT_* (negative: a name it does not know).
PyObject* matmul(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  if (nargs != 14 || abi.ws == nullptr) return none();
  if (!exact_tensor(a[0]) || !exact_tensor(a[1]) || !exact_tensor(a[2])) return none();
  const at::Tensor &x = THPVariable_Unpack(a[0]), &wq = THPVariable_Unpack(a[1]), &scales = THPVariable_Unpack(a[2]);
  int64_t bits, group, zero_point, kernel, activation, n;
  if (!take_int(a[3], &bits) || !take_int(a[4], &group) || !take_int(a[7], &kernel) || !take_int(a[10], &activation)) return none();
  if ((bits != 4 && bits != 8) || group <= 0 || group > (1 << 30) || activation < 0) return none();
  if (a[5] == Py_None) zero_point = bits == 4 ? 7 : 0;
  else if (!take_int(a[5], &zero_point) || zero_point < 0 || zero_point > 15) return none();
  if (!plain(x, at::kHalf) || x.dim() != 2 || !packed_words(wq) || !plain(scales, at::kHalf) || scales.dim() != 2) return none();
  const bool tiled = a[12] != Py_None;
  const int64_t m = x.size(0), k = x.size(1), words = k * bits / 32;
  if (!tiled) {
    n = wq.size(0);
  } else {
    if (!take_int(a[12], &n) || n < 0 || activation == MI355X_WQ_ACT_SILU_MUL) return none();
  }
  const int64_t rows = tiled ? (n + 15) / 16 * 16 : n;  // tile-major buffers hold whole tiles of rows
  if (k % 32 != 0 || k % group != 0 || wq.size(0) != rows || wq.size(1) != words || scales.size(0) != rows || scales.size(1) != k / group) return none();
  const int64_t out_cols = activation == MI355X_WQ_ACT_SILU_MUL ? n / 2 : n;

  mi355x_wq_epilogue ep{nullptr, nullptr, (int32_t)activation, 0};
  if (a[9] != Py_None) {
    if (!exact_tensor(a[9])) return none();
    const at::Tensor& b = THPVariable_Unpack(a[9]);
    if (!plain(b, at::kHalf) || b.numel() != n || !(b.dim() == 1 || (b.dim() == 2 && b.size(0) == 1))) return none();
    ep.bias = b.data_ptr();
  }
  if (a[11] != Py_None) {
    if (!exact_tensor(a[11])) return none();
    const at::Tensor& r = THPVariable_Unpack(a[11]);
    if (!plain(r, at::kHalf) || r.dim() != 2 || r.size(0) != m || r.size(1) != n) return none();
    ep.residual = r.data_ptr();
  }
  void* workspace = nullptr;
  int64_t workspace_bytes = 0;
  if (a[13] != Py_None) {
    if (!exact_tensor(a[13]) || kernel != 0) return none();
    const at::Tensor& w = THPVariable_Unpack(a[13]);
    if (!w.is_cuda() || !w.is_contiguous()) return none();
    workspace = w.data_ptr();
    workspace_bytes = (int64_t)w.nbytes();
  }
  void* stream = nullptr;
  if (!take_stream(a[8], &stream)) return none();

  const mi355x_wq_desc d{(int32_t)bits, (int32_t)group, (int32_t)zero_point, 0, n, k};
  const bool given = a[6] != Py_None;
  at::Tensor y;
  if (given) {
    if (!exact_tensor(a[6])) return none();
    y = THPVariable_Unpack(a[6]);
    if (!plain(y, at::kHalf) || y.dim() != 2 || y.size(0) != m || y.size(1) != out_cols) return none();
  }
  int rc = 0;
  bool failed = false;
  Py_BEGIN_ALLOW_THREADS
  try {
    if (!given) y = at::detail::empty_cuda({m, out_cols}, at::kHalf, x.device(), c10::nullopt);
    void* const py = y.data_ptr();
    if (workspace != nullptr) rc = abi.ws(&d, x.data_ptr(), wq.data_ptr(), scales.data_ptr(), &ep, py, m, stream, tiled ? 1 : 0, workspace, workspace_bytes);
    else if (tiled) rc = abi.tiled_ex(&d, x.data_ptr(), wq.data_ptr(), scales.data_ptr(), &ep, py, m, stream, (int)kernel);
    else rc = abi.fused_ex(&d, x.data_ptr(), wq.data_ptr(), scales.data_ptr(), &ep, py, m, stream, (int)kernel);
  } catch (...) {
    failed = true;  // (out of memory: the Python path allocates again and reports it)
  }
  Py_END_ALLOW_THREADS
  if (failed) return none();
  if (rc != 0) Py_RETURN_FALSE;
  if (given) {
    Py_INCREF(a[6]);
    return a[6];
  }
  return THPVariable_Wrap(std::move(y));
}

// dequantize(wq, scales, bits, group, zero_point, out, stream)
PyObject* dequantize(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  if (nargs != 7 || abi.dequantize == nullptr || !exact_tensor(a[0]) || !exact_tensor(a[1])) return none();
  const at::Tensor &wq = THPVariable_Unpack(a[0]), &scales = THPVariable_Unpack(a[1]);
  int64_t bits, group, zero_point;
  if (!take_int(a[2], &bits) || !take_int(a[3], &group) || (bits != 4 && bits != 8) || group <= 0 || group > (1 << 30)) return none();
  if (a[4] == Py_None) zero_point = bits == 4 ? 7 : 0;
  else if (!take_int(a[4], &zero_point) || zero_point < 0 || zero_point > 15) return none();
  if (!packed_words(wq) || !plain(scales, at::kHalf) || scales.dim() != 2 || a[5] != Py_None) return none();
  const int64_t n = wq.size(0), k = wq.size(1) * 32 / bits;
  if (scales.size(0) != n || scales.size(1) != k / group) return none();
  void* stream = nullptr;
  if (!take_stream(a[6], &stream)) return none();
  const mi355x_wq_desc d{(int32_t)bits, (int32_t)group, (int32_t)zero_point, 0, n, k};
  at::Tensor y;
  int rc = 0;
  bool failed = false;
  Py_BEGIN_ALLOW_THREADS
  try {
    y = at::detail::empty_cuda({n, k}, at::kHalf, wq.device(), c10::nullopt);
    rc = abi.dequantize(&d, wq.data_ptr(), scales.data_ptr(), y.data_ptr(), stream);
  } catch (...) {
    failed = true;
  }
  Py_END_ALLOW_THREADS
  if (failed) return none();
  if (rc != 0) Py_RETURN_FALSE;
  return THPVariable_Wrap(std::move(y));
}

// packed_call(function, resource, tensors): one call of a module's packed function with torch tensors, described as the
// caller of the boundary describes them (DLPack tensors without strides, int32 storage as packed uint32 words).
PyObject* packed_call(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  constexpr Py_ssize_t kMax = 8, kMaxDims = 8;
  if (nargs != 3 || !PyTuple_CheckExact(a[2])) return none();
  const Py_ssize_t n = PyTuple_GET_SIZE(a[2]);
  if (n > kMax) return none();
  mi355x_tvm_value values[kMax];
  int codes[kMax];
  mi355x_dl_tensor dl[kMax];
  int64_t shapes[kMax][kMaxDims];
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* const o = PyTuple_GET_ITEM(a[2], i);
    if (!exact_tensor(o)) return none();
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.is_cuda() || t.dim() > kMaxDims) return none();
    dl[i] = mi355x_dl_tensor{};
    if (t.scalar_type() == at::kHalf) dl[i].dtype.code = 2, dl[i].dtype.bits = 16;
    else if (t.scalar_type() == at::kInt || t.scalar_type() == at::kUInt32) dl[i].dtype.code = 1, dl[i].dtype.bits = 32;
    else return none();
    dl[i].dtype.lanes = 1;
    for (int64_t d = 0; d < t.dim(); ++d) shapes[i][d] = t.size(d);
    dl[i].data = t.data_ptr();
    dl[i].device.device_type = MI355X_DL_ROCM;
    dl[i].device.device_id = t.device().index();
    dl[i].ndim = (int32_t)t.dim();
    dl[i].shape = shapes[i];
    values[i].v_handle = &dl[i];
    codes[i] = MI355X_TVM_NDARRAY_HANDLE;
  }
  const auto fn = reinterpret_cast<mi355x_wq_packed_cfunc>(PyLong_AsVoidPtr(a[0]));
  void* const resource = PyLong_AsVoidPtr(a[1]);
  if (fn == nullptr || PyErr_Occurred()) {
    PyErr_Clear();
    return none();
  }
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = fn(values, codes, (int)n, nullptr, resource);
  Py_END_ALLOW_THREADS
  if (rc != 0) Py_RETURN_FALSE;
  Py_RETURN_TRUE;
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject* self, PyObject* const* a, Py_ssize_t nargs) {
  try {
    return F(self, a, nargs);
  } catch (...) {
    PyErr_Clear();
    return none();
  }
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyCFunction entry() {
  return reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&guarded<F>));
}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    {"matmul", entry<matmul>(), METH_FASTCALL, nullptr},
    {"dequantize", entry<dequantize>(), METH_FASTCALL, nullptr},
    {"packed_call", entry<packed_call>(), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_wq_torch", "native host path of relax_amd", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__wq_torch(void) { return PyModule_Create(&module_def); }
