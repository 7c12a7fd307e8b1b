// The three linears of ops.py from their tensors to the launch in one native call.
//
// A small call is bound by the host: a decode GEMV of N = K = 4096 runs 3.6 us on the device, and checking the operands,
// allocating the result and converting ten arguments in Python took 7.4 us.  Here the common form of a call (plain device
// tensors of the right types and shapes, no mode that wants to see the single steps) takes what is measured beside the
// functions in ops.py.  Everything else, errors included, is answered with None: the caller then goes through its own
// checks, which say what is wrong or take the call as they always did.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TracerMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../../include/relax_amd_wq.h"

namespace {

struct {
  decltype(&wq_q4g32_linear) q4g32_linear;
  decltype(&wq_fpA_intB_gemm) intb;
  decltype(&wq_fpA_intB_gemm_residual) intb_residual;
  decltype(&wq_gptq_linear) gptq_linear;
  decltype(&wq_gptq_workspace_bytes) gptq_workspace_bytes;
  PyObject *device, *stream;  // torch._C._cuda_getDevice, torch._C._cuda_getCurrentRawStream
} g;

// nobody watches the steps of this call: no function or dispatch mode, no tracing
bool unwatched() {
  return g.q4g32_linear && !at::impl::torch_function_mode_enabled() && !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
         !at::tracer::impl::is_dispatch_enabled();
}

struct Operand {
  const at::Tensor* t = nullptr;
  void* p = nullptr;  // stays null for an operand that is None
};

bool device_tensor(PyObject* o, Operand& r) {
  if (!THPVariable_CheckExact(o)) return false;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || t.layout() != at::kStrided || !t.has_storage() || t.unsafeGetTensorImpl()->is_python_dispatch() ||
      !t.is_cuda() || !t.is_contiguous() || t.numel() == 0)
    return false;
  r.t = &t;
  r.p = t.data_ptr();
  return true;
}
bool typed(PyObject* o, at::ScalarType type, Operand& r) { return device_tensor(o, r) && r.t->scalar_type() == type; }
bool half_or_none(PyObject* o, Operand& r) { return o == Py_None || typed(o, at::kHalf, r); }
bool holds(const Operand& r, int64_t numel) { return !r.t || r.t->numel() == numel; }

bool current_stream(wq_stream_t* s) {
  PyObject* dev = PyObject_CallNoArgs(g.device);
  PyObject* raw = dev ? PyObject_CallOneArg(g.stream, dev) : nullptr;
  Py_XDECREF(dev);
  if (!raw) return false;
  *s = (wq_stream_t)PyLong_AsVoidPtr(raw);
  Py_DECREF(raw);
  return !PyErr_Occurred();
}

struct WithoutGil {
  PyThreadState* state = PyEval_SaveThread();
  ~WithoutGil() { PyEval_RestoreThread(state); }
};

// what x is multiplied into: [..., N]
at::Tensor result_like(const at::Tensor& x, int64_t N) {
  c10::SmallVector<int64_t, 6> sizes(x.sizes().begin(), x.sizes().end());
  sizes.back() = N;
  return at::empty(sizes, x.options());
}

// `launch(y, stream)` into a new tensor, or into `out` where one is given; a new reference, or null: not done
template <class Launch>
PyObject* launched(const Operand& x, int64_t N, PyObject* out, Launch launch) {
  Operand y;
  wq_stream_t stream;
  if (out != Py_None && (!typed(out, at::kHalf, y) || !holds(y, x.t->numel() / x.t->size(-1) * N))) return nullptr;
  if (!current_stream(&stream)) return nullptr;
  at::Tensor made;
  int rc;
  {
    WithoutGil released;
    if (!y.t) made = result_like(*x.t, N);
    rc = launch(y.t ? y.p : made.data_ptr(), stream);
  }
  if (rc != WQ_OK) return nullptr;
  if (!y.t) return THPVariable_Wrap(std::move(made));
  Py_INCREF(out);
  return out;
}

template <class Call>
PyObject* or_none(Call call) {
  PyObject* r = nullptr;
  try {
    if (unwatched()) r = call();
  } catch (...) {
    r = nullptr;
  }
  if (r) return r;
  PyErr_Clear();
  Py_RETURN_NONE;
}

#define U16(o) ((const uint16_t*)(o).p)

// (W, S, x, bias, residual, out)
PyObject* q4g32_linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return or_none([&]() -> PyObject* {
    Operand W, S, x, bias, residual;
    if (n != 6 || !device_tensor(a[0], W) || !typed(a[1], at::kHalf, S) || !typed(a[2], at::kHalf, x) ||
        !half_or_none(a[3], bias) || !half_or_none(a[4], residual))
      return nullptr;
    if ((W.t->scalar_type() != at::kInt && W.t->scalar_type() != at::kUInt32) || W.t->dim() != 2 || S.t->dim() != 2 || x.t->dim() < 1)
      return nullptr;
    const int64_t N = W.t->size(0), K = W.t->size(1) * 8, M = x.t->numel() / K;
    if (x.t->size(-1) != K || K % 32 || S.t->size(0) != N || S.t->size(1) != K / 32 || !holds(bias, N) || !holds(residual, M * N))
      return nullptr;
    return launched(x, N, a[5], [&](void* y, wq_stream_t stream) {
      return g.q4g32_linear((const uint32_t*)W.p, U16(S), U16(x), U16(bias), U16(residual), (uint16_t*)y, M, N, K, stream);
    });
  });
}

// (x, B, scales, bias, residual, bits, activation, binary, unary, group size, out)
PyObject* fpA_intB_gemm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return or_none([&]() -> PyObject* {
    Operand x, B, scales, bias, residual;
    if (n != 11 || !typed(a[0], at::kHalf, x) || !typed(a[1], at::kChar, B) || !typed(a[2], at::kHalf, scales) ||
        !half_or_none(a[3], bias) || !half_or_none(a[4], residual))
      return nullptr;
    int64_t v[5];
    for (int i = 0; i < 5; ++i) {
      if (!PyLong_CheckExact(a[5 + i])) return nullptr;
      v[i] = PyLong_AsLongLong(a[5 + i]);
      if (v[i] == -1 && PyErr_Occurred()) return nullptr;
    }
    const int64_t bits = v[0], group = v[4];
    if ((bits != 4 && bits != 8) || B.t->dim() != 2 || x.t->dim() < 1) return nullptr;
    const int64_t K = B.t->size(0), N = B.t->size(1) * (bits == 4 ? 2 : 1), M = x.t->numel() / K;
    const int64_t want = group <= 0 || group == K ? N : (K / group) * N;
    if (x.t->size(-1) != K || scales.t->numel() != want || !holds(bias, N) || (bias.t && (bias.t->dim() < 1 || bias.t->size(-1) != N)) ||
        !holds(residual, M * N))
      return nullptr;
    return launched(x, N, a[10], [&](void* y, wq_stream_t stream) {
      if (!residual.t)
        return g.intb(U16(x), (const int8_t*)B.p, U16(scales), U16(bias), (uint16_t*)y, (int)v[1], M, N, K, group, 0, (int)bits,
                      nullptr, 0, stream);
      return g.intb_residual(U16(x), (const int8_t*)B.p, U16(scales), U16(bias), U16(residual), (uint16_t*)y, (int)v[1], (int)v[2],
                             (int)v[3], M, N, K, group, (int)bits, nullptr, 0, stream);
    });
  });
}

// (W_nk, SZ, perm, x, bias, residual, N, K, groups)
PyObject* gptq_linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return or_none([&]() -> PyObject* {
    Operand W, SZ, perm, x, bias, residual;
    if (n != 9 || !device_tensor(a[0], W) || !device_tensor(a[1], SZ) || !(a[2] == Py_None || device_tensor(a[2], perm)) ||
        !typed(a[3], at::kHalf, x) || !half_or_none(a[4], bias) || !half_or_none(a[5], residual))
      return nullptr;
    int64_t v[3];
    for (int i = 0; i < 3; ++i) {
      if (!PyLong_CheckExact(a[6 + i])) return nullptr;
      v[i] = PyLong_AsLongLong(a[6 + i]);
      if (v[i] <= 0) return nullptr;
    }
    const int64_t N = v[0], K = v[1], M = x.t->numel() / K;
    if (x.t->dim() < 1 || x.t->size(-1) != K || (bias.t && bias.t->numel() < N) || !holds(residual, M * N)) return nullptr;
    return launched(x, N, Py_None, [&](void* y, wq_stream_t stream) {
      const size_t need = g.gptq_workspace_bytes(M, K, perm.t != nullptr);
      at::Tensor space;
      if (need) space = at::empty({(int64_t)need}, x.t->options().dtype(at::kByte));
      return g.gptq_linear((const uint32_t*)W.p, U16(SZ), (const int32_t*)perm.p, U16(x), U16(bias), U16(residual), (uint16_t*)y,
                           M, N, K, v[2], need ? space.data_ptr() : nullptr, need, stream);
    });
  });
}

// (addresses of the five entry points, torch's two functions)
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 7) {
    PyErr_SetString(PyExc_TypeError, "bind takes five addresses and two functions");
    return nullptr;
  }
  void* p[5];
  for (int i = 0; i < 5; ++i) {
    p[i] = PyLong_AsVoidPtr(a[i]);
    if (PyErr_Occurred()) return nullptr;
  }
  Py_INCREF(a[5]);
  Py_INCREF(a[6]);
  g.device = a[5], g.stream = a[6];
  g.intb = (decltype(g.intb))p[1];
  g.intb_residual = (decltype(g.intb_residual))p[2];
  g.gptq_linear = (decltype(g.gptq_linear))p[3];
  g.gptq_workspace_bytes = (decltype(g.gptq_workspace_bytes))p[4];
  g.q4g32_linear = (decltype(g.q4g32_linear))p[0];
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void*)bind, METH_FASTCALL, nullptr},
    {"q4g32_linear", (PyCFunction)(void*)q4g32_linear, METH_FASTCALL, nullptr},
    {"fpA_intB_gemm", (PyCFunction)(void*)fpA_intB_gemm, METH_FASTCALL, nullptr},
    {"gptq_linear", (PyCFunction)(void*)gptq_linear, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls() {
  PyObject* m = PyModule_Create(&module);
  // (its layout of a tensor is that of this torch and of no other)
  if (m && PyModule_AddStringConstant(m, "torch_version", RELAX_AMD_TORCH_VERSION) != 0) Py_CLEAR(m);
  return m;
}
