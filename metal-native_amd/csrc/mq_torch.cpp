// Native front of the small calls: dequant_matmul and the fp16 / fp32 vecmat
// route of matmul on plain torch tensors, as one CPython call.
//
// Why: a decode GEMV of a small layer runs 4-9 us on the GPU, and the Python
// checks, the allocation and the ctypes call around it took 15 us on the host
// (vecmat: 17).  Here the same checks, the output's allocation and the launch
// take 4.8 us (K = 896, N = 4864, M = 1 called in a row: 13.3 -> 5.7 us).
//
// Only the plain case is taken: exact torch tensors (no subclass, no
// dispatch or function mode, no lazy negation) in row-major layouts that the
// kernels address directly and arguments that ops.py would accept.  For
// anything else the functions return None and ops.py goes its general way,
// which copies, or raises its errors.  An error of the library comes back as
// its code (an int).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/metal_native_amd.h"

namespace {

bool modes_set() { return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled(); }

// a strided GPU tensor with memory of its own and nothing pending on it
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || at::isTensorSubclassLike(t) || t.is_neg() ||
      t._is_zerotensor() || !t.has_storage())
    return nullptr;
  return &t;
}

// 2-D, rows of unit stride that do not overlap
bool rowmajor(const at::Tensor& t) {
  return t.dim() == 2 && (t.size(1) <= 1 || t.stride(1) == 1) && (t.size(0) <= 1 || t.stride(0) >= t.size(1));
}
int64_t ld(const at::Tensor& t) { return t.size(0) > 1 ? t.stride(0) : t.size(1); }

PyObject* decline() { Py_RETURN_NONE; }

// (activations, weights, scales, zeros, group_size, is_int4, epilogue code, bias | None, residual | None, stream)
PyObject* dequant_matmul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 10) {
    PyErr_SetString(PyExc_TypeError, "dequant_matmul: 10 arguments");
    return nullptr;
  }
  if (modes_set()) return decline();
  const at::Tensor *x = plain(a[0]), *w = plain(a[1]), *s = plain(a[2]), *z = plain(a[3]);
  if (!x || !w || !s || !z || !PyLong_CheckExact(a[4])) return decline();
  int over = 0;
  const int64_t g = PyLong_AsLongLongAndOverflow(a[4], &over);
  const bool int4 = a[5] == Py_True;
  const int epi = (int)PyLong_AsLong(a[6]);
  if (over || PyErr_Occurred()) {
    PyErr_Clear();
    return decline();
  }
  if (!rowmajor(*x) || !rowmajor(*w)) return decline();
  const int64_t M = x->size(0), K = x->size(1), N = w->size(0);
  const c10::Device dev = x->device();
  if (M < 1 || N < 1 || K < 1 || x->scalar_type() != at::kHalf || w->device() != dev || s->device() != dev ||
      z->device() != dev || (w->scalar_type() != at::kByte && w->scalar_type() != at::kChar) ||
      s->scalar_type() != at::kHalf || z->scalar_type() != at::kHalf)
    return decline();
  if (!(g == 32 || g == 64 || g == 128 || g == K)) return decline();
  if (int4 ? (K % 2 != 0 || w->size(1) != K / 2) : w->size(1) != K) return decline();
  const int64_t G = (K + g - 1) / g;
  for (const at::Tensor* t : {s, z})
    if (t->dim() != 2 || t->size(0) != N || t->size(1) != G || !t->is_contiguous()) return decline();
  const void *bias = nullptr, *resid = nullptr;
  int64_t ldr = 0;
  const bool wants_bias = epi == MQ_EPILOGUE_BIAS || epi == MQ_EPILOGUE_BIAS_RELU || epi == MQ_EPILOGUE_BIAS_SILU;
  if (wants_bias != (a[7] != Py_None) || (epi == MQ_EPILOGUE_RESIDUAL) != (a[8] != Py_None)) return decline();
  if (epi < MQ_EPILOGUE_NONE || epi > MQ_EPILOGUE_SWIGLU || (epi == MQ_EPILOGUE_SWIGLU && N % 2)) return decline();
  if (wants_bias) {
    const at::Tensor* b = plain(a[7]);
    if (!b || b->device() != dev || b->scalar_type() != at::kHalf || b->numel() != N || !b->is_contiguous()) return decline();
    bias = b->const_data_ptr();
  }
  if (epi == MQ_EPILOGUE_RESIDUAL) {
    const at::Tensor* r = plain(a[8]);
    if (!r || r->device() != dev || r->scalar_type() != at::kHalf || !rowmajor(*r) || r->size(0) != M || r->size(1) != N)
      return decline();
    resid = r->const_data_ptr();
    ldr = ld(*r);
  }
  const int64_t nout = epi == MQ_EPILOGUE_SWIGLU ? N / 2 : N;
  void* stream = PyLong_AsVoidPtr(a[9]);
  if (PyErr_Occurred()) return nullptr;
  HANDLE_TH_ERRORS
  const c10::DeviceGuard guard(dev);
  at::Tensor out = at::empty({M, nout}, x->options());
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = mq_dequant_matmul(x->const_data_ptr(), ld(*x), w->const_data_ptr(), ld(*w), s->const_data_ptr(),
                         z->const_data_ptr(), out.mutable_data_ptr(), nout, M, N, K, (int32_t)g,
                         int4 ? MQ_QUANT_INT4 : MQ_QUANT_INT8, epi, bias, resid, ldr, stream);
  Py_END_ALLOW_THREADS
  return rc == MQ_SUCCESS ? THPVariable_Wrap(std::move(out)) : PyLong_FromLong(rc);
  END_HANDLE_TH_ERRORS
}

// (a, b, transpose_b, stream): a [M <= 8, K], b [K, N] or [N, K], N, K >= 256
PyObject* vecmat(PyObject*, PyObject* const* p, Py_ssize_t n) {
  if (n != 4) {
    PyErr_SetString(PyExc_TypeError, "vecmat: 4 arguments");
    return nullptr;
  }
  if (modes_set()) return decline();
  const at::Tensor *a = plain(p[0]), *b = plain(p[1]);
  if (!a || !b || !rowmajor(*a) || !rowmajor(*b)) return decline();
  const bool tb = p[2] == Py_True;
  const int64_t M = a->size(0), K = a->size(1), N = tb ? b->size(0) : b->size(1);
  const c10::Device dev = a->device();
  const at::ScalarType ty = a->scalar_type();
  if (b->device() != dev || b->scalar_type() != ty || (ty != at::kHalf && ty != at::kFloat) ||
      (tb ? b->size(1) : b->size(0)) != K || M < 1 || M > 8 || N < 256 || K < 256)
    return decline();
  void* stream = PyLong_AsVoidPtr(p[3]);
  if (PyErr_Occurred()) return nullptr;
  HANDLE_TH_ERRORS
  const c10::DeviceGuard guard(dev);
  at::Tensor out = at::empty({M, N}, a->options());
  const auto fn = ty == at::kHalf ? mq_vecmat_f16 : mq_vecmat_f32;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = fn(a->const_data_ptr(), ld(*a), b->const_data_ptr(), ld(*b), out.mutable_data_ptr(), N, M, N, K, tb ? 1 : 0,
          stream);
  Py_END_ALLOW_THREADS
  return rc == MQ_SUCCESS ? THPVariable_Wrap(std::move(out)) : PyLong_FromLong(rc);
  END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"dequant_matmul", (PyCFunction)(void (*)(void))dequant_matmul, METH_FASTCALL, nullptr},
    {"vecmat", (PyCFunction)(void (*)(void))vecmat, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_mq_torch", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__mq_torch(void) { return PyModule_Create(&kModule); }
