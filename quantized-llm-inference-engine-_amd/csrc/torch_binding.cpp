// The per-call host path of a packed linear, in native code: checks the plain form of a call (contiguous
// tensors of the expected dtypes and shapes on one device), allocates the output and the workspace from
// torch's caching allocator and calls the C ABI on the current stream. The checks run on every call and
// nothing is kept between calls. A call in any other form returns None, and the caller takes the general
// path, which converts, broadcasts or raises as torch would.
//
// Why: at one token the kernel takes 4.8 us, and the same steps in Python (attribute look-ups, checks,
// two ctypes calls) held a 4096 x 4096 call at 18.9 us; 6.9 us with this path.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <pybind11/pybind11.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

namespace {

using LinearFn = int (*)(const void*, int64_t, int64_t, int64_t, const void*, int64_t, const float*, const float*,
                         const void*, void*, int64_t, int64_t, int, int, int, int, int, void*, size_t, void*, int);
using SwigluFn = int (*)(const void*, int64_t, int64_t, int64_t, const void*, int64_t, const float*, const float*,
                         const void*, void*, int64_t, int64_t, int, int, int, int, int, void*, size_t, void*);
using WorkspaceFn = size_t (*)(int64_t, int64_t, int64_t, int, int, int);

struct Api {
  LinearFn linear = nullptr;
  SwigluFn swiglu = nullptr;
  WorkspaceFn linear_ws = nullptr, swiglu_ws = nullptr;
} g_api;

// attach(linear_ex, linear_workspace_ex, linear_swiglu, linear_swiglu_workspace_ex): the C ABI's addresses.
PyObject* attach(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 4) {
    PyErr_SetString(PyExc_TypeError, "attach takes four addresses");
    return nullptr;
  }
  void* p[4];
  for (int i = 0; i < 4; ++i) {
    p[i] = PyLong_AsVoidPtr(args[i]);
    if (!p[i] && PyErr_Occurred()) return nullptr;
  }
  g_api.linear = reinterpret_cast<LinearFn>(p[0]);
  g_api.linear_ws = reinterpret_cast<WorkspaceFn>(p[1]);
  g_api.swiglu = reinterpret_cast<SwigluFn>(p[2]);
  g_api.swiglu_ws = reinterpret_cast<WorkspaceFn>(p[3]);
  Py_RETURN_NONE;
}

const at::Tensor* tensor_of(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

// linear(x, qweight, scales, zeros, bias, out_features, in_features, bits, group_size, symmetric, dtype,
// swiglu) -> tensor or None. dtype: 0 fp32, 1 fp16, 2 bf16. swiglu: fused gate/up rows, out_features / 2
// columns come back.
PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 12 || !g_api.linear) {
    PyErr_SetString(PyExc_TypeError, "linear takes twelve arguments, after attach");
    return nullptr;
  }
  HANDLE_TH_ERRORS  // torch's own exception types: an allocation that fails is torch.OutOfMemoryError
  if (!THPVariable_CheckExact(args[0])) Py_RETURN_NONE;  // a subclass may see the general path's torch calls
  const at::Tensor *x = tensor_of(args[0]), *qw = tensor_of(args[1]), *sc = tensor_of(args[2]);
  const at::Tensor* zp = tensor_of(args[3]);
  const at::Tensor* bias = tensor_of(args[4]);
  if (!x || !qw || !sc || (!bias && args[4] != Py_None)) Py_RETURN_NONE;
  int64_t v[7];
  for (int i = 0; i < 7; ++i) {
    v[i] = PyLong_AsLongLong(args[5 + i]);
    if (v[i] == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      Py_RETURN_NONE;
    }
  }
  const int64_t N = v[0], K = v[1], bits = v[2], group = v[3] > 0 ? v[3] : v[1], dtype = v[5];
  const bool symmetric = v[4] != 0, swiglu = v[6] != 0;
  if (N < 1 || K < 1 || N > INT32_MAX || K > INT32_MAX || bits < 1 || bits > 8 || K % group != 0 || dtype < 0 ||
      dtype > 2 || (swiglu && N % 8 != 0))
    Py_RETURN_NONE;
  const at::ScalarType act = dtype == 0 ? at::kFloat : dtype == 1 ? at::kHalf : at::kBFloat16;
  const at::Device dev = x->device();
  if (!dev.is_cuda() || x->layout() != at::kStrided || x->scalar_type() != act || x->dim() < 1 ||
      x->size(-1) != K || !x->is_contiguous())
    Py_RETURN_NONE;
  const int64_t G = K / group, M = x->numel() / K;
  if (M < 1) Py_RETURN_NONE;
  const bool is_signed = qw->scalar_type() == at::kChar;
  if (qw->device() != dev || !(qw->scalar_type() == at::kByte || (bits == 8 && is_signed)) || qw->dim() != 2 ||
      qw->size(0) != N || qw->size(1) < (bits == 8 ? K : (K + 1) / 2) || !qw->is_contiguous())
    Py_RETURN_NONE;
  auto plain_meta = [&](const at::Tensor* t) {
    return t && t->device() == dev && t->scalar_type() == at::kFloat && t->dim() == 2 && t->size(0) == N &&
           t->size(1) == G && t->is_contiguous();
  };
  if (!plain_meta(sc) || (!symmetric && !plain_meta(zp))) Py_RETURN_NONE;
  if (bias && (bias->device() != dev || bias->scalar_type() != act || bias->dim() != 1 || bias->size(0) != N ||
               !bias->is_contiguous()))
    Py_RETURN_NONE;

  const size_t ws_bytes = (swiglu ? g_api.swiglu_ws : g_api.linear_ws)(M, N, K, int(bits), int(group), int(dtype));
  const int64_t cols = swiglu ? N / 2 : N;
  at::Tensor y, ws;
  {
    const auto options = at::TensorOptions().device(dev);
    c10::SmallVector<int64_t, 6> shape(x->sizes().begin(), x->sizes().end());
    shape.back() = cols;
    y = at::empty(shape, options.dtype(act));
    if (ws_bytes) ws = at::empty({int64_t(ws_bytes)}, options.dtype(at::kByte));
  }
  void* stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
  const void *xp = x->const_data_ptr(), *qp = qw->const_data_ptr();
  const float *sp = sc->const_data_ptr<float>(), *zpp = symmetric ? nullptr : zp->const_data_ptr<float>();
  const void* bp = bias ? bias->const_data_ptr() : nullptr;
  void *yp = y.mutable_data_ptr(), *wp = ws_bytes ? ws.mutable_data_ptr() : nullptr;
  int rc;
  {
    pybind11::gil_scoped_release released;  // taken again also where the call throws
    rc = swiglu ? g_api.swiglu(xp, M, K, K, qp, qw->size(1), sp, zpp, bp, yp, N, cols, int(dtype), int(bits),
                               int(group), symmetric, is_signed, wp, ws_bytes, stream)
                : g_api.linear(xp, M, K, K, qp, qw->size(1), sp, zpp, bp, yp, N, cols, int(dtype), int(bits),
                               int(group), symmetric, is_signed, wp, ws_bytes, stream, 0);
  }
  if (rc != 0) Py_RETURN_NONE;  // the general path asks again and reports the error
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"attach", reinterpret_cast<PyCFunction>(attach), METH_FASTCALL, nullptr},
    {"linear", reinterpret_cast<PyCFunction>(linear), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_llmopt_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__llmopt_torch(void) {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) != 0) Py_CLEAR(m);
  return m;
}
