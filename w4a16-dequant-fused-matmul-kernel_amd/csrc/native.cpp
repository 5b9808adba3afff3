// _native: the automatic GEMM call as one C function of the CPython API, for the
// ordinary call (plain strided HIP tensors on the current device, zeros already
// checked, autotuning off).  Anything else -- wrong types, shapes, layouts or
// devices, tensor subclasses, functorch wrappers, dispatch modes, an unchecked
// zeros tensor, an empty result -- returns None, and the caller's Python path
// checks, raises or computes as it always has.
//
// The same call through Python's checks, context managers and ctypes took 13-20
// us on the host, more than most decode and small-batch kernels run: repeated
// calls at M = 1, K = N = 1024 went from 13.5 to 4.9 us each, W4A16Linear at
// 1 x 4096 x 4096 from 18.1 to 5.8, at 8 x 4096 x 6144 from 18.5 to 6.0.  Nothing
// is kept between calls: the split-K workspace comes from torch's caching
// allocator, whose blocks follow the stream they were allocated on (and, under
// graph capture, belong to the graph).
#include <Python.h>
#include <dlfcn.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/w4a16.h"

#ifndef W4A16_NATIVE_HASH
#define W4A16_NATIVE_HASH "unknown"
#endif

namespace {

decltype(&w4a16_gemm_f16_auto) g_gemm = nullptr;
decltype(&w4a16_gemm_workspace_bytes) g_workspace = nullptr;
PyObject* g_zeros_key = nullptr;   // interned attribute name of the zeros check

constexpr int64_t kGroupMultiple = 32;

// A plain dense tensor this code may read: no subclass, no functorch, functional,
// fake or Python-dispatched wrapper.
bool plain(PyObject* o, const at::Tensor** t) {
  if (!THPVariable_CheckExact(o)) return false;
  const at::Tensor& v = THPVariable_Unpack(o);
  if (!v.defined() || !v.is_cuda() || v.layout() != at::kStrided || !v.has_storage()) return false;
  const auto ks = v.key_set();
  using K = c10::DispatchKey;
  if (ks.has_any(c10::DispatchKeySet({K::Python, K::PythonTLSSnapshot, K::FuncTorchBatched,
                                      K::FuncTorchGradWrapper, K::BatchedNestedTensor,
                                      K::Functionalize, K::Negative, K::Conjugate, K::ZeroTensor})))
    return false;
  *t = &v;
  return true;
}

bool rows_ok(const at::Tensor& t) {
  return t.is_contiguous() ||
         (t.dim() == 2 && t.stride(1) == 1 && t.stride(0) >= t.size(1));
}
int64_t row_stride(const at::Tensor& t) { return t.size(0) > 1 ? t.stride(0) : t.size(1); }

// The zeros check's result kept on the tensor object (hip_kernel.py): the tuple
// ((version, data_ptr, numel, device), need), still valid for the tensor as it
// is now.  -1: none or outdated.
int checked_zeros(PyObject* o, const at::Tensor& z) {
  if (z.is_inference()) return -1;
  // (straight from its dict: a missing attribute's exception costs a weight's first
  // call 0.5 us)
  PyObject** dict = _PyObject_GetDictPtr(o);
  PyObject* hit = dict && *dict ? PyDict_GetItemWithError(*dict, g_zeros_key) : nullptr;
  if (!hit) {
    PyErr_Clear();
    return -1;
  }
  Py_INCREF(hit);
  int need = -1;
  if (PyTuple_CheckExact(hit) && PyTuple_GET_SIZE(hit) == 2) {
    PyObject *key = PyTuple_GET_ITEM(hit, 0), *flag = PyTuple_GET_ITEM(hit, 1);
    if (PyTuple_CheckExact(key) && PyTuple_GET_SIZE(key) == 4) {
      // (the device is part of the storage's address)
      const int64_t version = PyLong_AsLongLong(PyTuple_GET_ITEM(key, 0));
      const uint64_t ptr = PyLong_AsUnsignedLongLong(PyTuple_GET_ITEM(key, 1));
      const int64_t numel = PyLong_AsLongLong(PyTuple_GET_ITEM(key, 2));
      if (PyErr_Occurred())
        PyErr_Clear();
      else if (version == (int64_t)z._version() && numel == z.numel() &&
               ptr == reinterpret_cast<uint64_t>(z.data_ptr()))
        need = flag == Py_True ? 1 : flag == Py_False ? 0 : -1;
    }
  }
  Py_DECREF(hit);
  return need;
}

// Something other than plain execution is on: a mode, a trace, a functorch
// transform.  The Python path runs under it as it did.
bool observed() {
  using K = c10::DispatchKey;
  const auto in = c10::impl::tls_local_dispatch_key_set().included_;
  return at::impl::torch_function_mode_enabled() ||
         c10::impl::TorchDispatchModeTLS::any_modes_set() ||
         in.has_any(c10::DispatchKeySet({K::Tracer, K::Functionalize, K::Python,
                                         K::PythonTLSSnapshot, K::FuncTorchBatched,
                                         K::FuncTorchVmapMode, K::FuncTorchDynamicLayerFrontMode,
                                         K::FuncTorchDynamicLayerBackMode}));
}

// gemm(x, qweight, scales, zeros, bias | None, group_size, out | None,
//      in_features | None, out_features): y, or None.  With in_features (a
// W4A16Linear's forward) x may have any number of dimensions, the result keeps
// all but the last, and the weight must be [in_features, out_features]; without
// it x is 2-D.
PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 9 || !g_gemm) Py_RETURN_NONE;
  const at::Tensor *x, *qw, *s, *z, *bias = nullptr, *out = nullptr;
  if (!plain(args[0], &x) || !plain(args[1], &qw) || !plain(args[2], &s) || !plain(args[3], &z) ||
      (args[4] != Py_None && !plain(args[4], &bias)) ||
      (args[6] != Py_None && !plain(args[6], &out)) || !PyLong_CheckExact(args[5]))
    Py_RETURN_NONE;
  if (observed()) Py_RETURN_NONE;
  const bool lead = args[7] != Py_None;
  if (lead && (!PyLong_CheckExact(args[7]) || !PyLong_CheckExact(args[8]))) Py_RETURN_NONE;
  const int64_t G = PyLong_AsLongLong(args[5]);
  const int64_t in_features = lead ? PyLong_AsLongLong(args[7]) : 0;
  const int64_t out_features = lead ? PyLong_AsLongLong(args[8]) : 0;
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const auto dev = x->device();
  if (x->scalar_type() != at::kHalf || qw->scalar_type() != at::kInt ||
      s->scalar_type() != at::kHalf || z->scalar_type() != at::kHalf || qw->dim() != 2 ||
      s->dim() != 2 || z->dim() != 2 || qw->device() != dev || s->device() != dev ||
      z->device() != dev || c10::hip::current_device() != dev.index())
    Py_RETURN_NONE;
  const int64_t K = qw->size(0) * 8, N = qw->size(1);
  if (G <= 0 || K == 0 || N == 0 || K % G != 0 || G % kGroupMultiple != 0 ||
      s->size(0) != K / G || s->size(1) != N || z->size(0) != K / G || z->size(1) != N ||
      !qw->is_contiguous() || !s->is_contiguous() || !z->is_contiguous())
    Py_RETURN_NONE;
  int64_t M, ldx;
  if (lead && x->dim() != 2) {
    if (x->dim() < 1 || x->size(-1) != K || !x->is_contiguous()) Py_RETURN_NONE;
    M = x->numel() / K;
    ldx = K;
  } else {
    if (x->dim() != 2 || x->size(1) != K || !rows_ok(*x)) Py_RETURN_NONE;
    M = x->size(0);
    ldx = row_stride(*x);
  }
  if (M == 0 || (lead && (in_features != K || out_features != N))) Py_RETURN_NONE;
  if (bias && (bias->dim() != 1 || bias->size(0) != N || bias->scalar_type() != at::kHalf ||
               !bias->is_contiguous() || bias->device() != dev))
    Py_RETURN_NONE;
  int64_t ldy = N;
  if (out) {
    if (out->dim() != 2 || out->size(0) != M || out->size(1) != N ||
        out->scalar_type() != at::kHalf || !rows_ok(*out) || out->device() != dev)
      Py_RETURN_NONE;
    ldy = row_stride(*out);
  }
  const int need = checked_zeros(args[3], *z);
  if (need < 0) Py_RETURN_NONE;

  at::Tensor y;
  if (!out) {
    if (lead && x->dim() != 2) {
      std::vector<int64_t> shape(x->sizes().begin(), x->sizes().end());
      shape.back() = N;
      y = at::empty(shape, at::TensorOptions().dtype(at::kHalf).device(dev));
    } else {
      y = at::empty({M, N}, at::TensorOptions().dtype(at::kHalf).device(dev));
    }
  }
  const size_t bytes = g_workspace(M, N, K, G);
  at::Tensor ws;
  if (bytes)
    ws = at::empty({(int64_t)bytes}, at::TensorOptions().dtype(at::kByte).device(dev));
  void* stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
  void *xp = x->data_ptr(), *qp = qw->data_ptr(), *sp = s->data_ptr(), *zp = z->data_ptr();
  void* bp = bias ? bias->data_ptr() : nullptr;
  void* yp = out ? out->data_ptr() : y.data_ptr();
  void* wp = bytes ? ws.data_ptr() : nullptr;
  int code;
  Py_BEGIN_ALLOW_THREADS
  code = g_gemm(xp, ldx, static_cast<const int32_t*>(qp), sp, zp, bp, yp, ldy, M, N, K, G,
                need ? W4A16_PLAN_ANY_ZEROS : 0, wp, bytes, stream);
  Py_END_ALLOW_THREADS
  if (code != W4A16_OK) Py_RETURN_NONE;   // the Python path repeats the call and raises
  if (out) {
    Py_INCREF(args[6]);
    return args[6];
  }
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// init(path of the loaded libw4a16.so, name of the zeros check's attribute)
PyObject* init(PyObject*, PyObject* args) {
  const char *path, *key;
  if (!PyArg_ParseTuple(args, "ss", &path, &key)) return nullptr;
  void* lib = dlopen(path, RTLD_NOW | RTLD_LOCAL);
  if (!lib) {
    PyErr_Format(PyExc_ImportError, "cannot open %s: %s", path, dlerror());
    return nullptr;
  }
  g_gemm = reinterpret_cast<decltype(g_gemm)>(dlsym(lib, "w4a16_gemm_f16_auto"));
  g_workspace = reinterpret_cast<decltype(g_workspace)>(dlsym(lib, "w4a16_gemm_workspace_bytes"));
  if (!g_gemm || !g_workspace) {
    g_gemm = nullptr;
    PyErr_Format(PyExc_ImportError, "%s lacks w4a16_gemm_f16_auto", path);
    return nullptr;
  }
  g_zeros_key = PyUnicode_InternFromString(key);
  if (!g_zeros_key) return nullptr;
  Py_RETURN_NONE;
}

PyObject* build_id(PyObject*, PyObject*) { return PyUnicode_FromString(W4A16_NATIVE_HASH); }

PyMethodDef kMethods[] = {
    {"gemm", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(gemm)), METH_FASTCALL,
     "The automatic GEMM call, or None where the Python path has to make it."},
    {"init", init, METH_VARARGS, "Bind the loaded libw4a16.so."},
    {"build_id", build_id, METH_NOARGS, "sha256 of the sources this module was built from."},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&kModule); }
