// The calls of the Python package from tensors to the C ABI, in native code.
//
// A decode or verify layer's kernel takes 3-20 us, and the Python form of a call (argument checks,
// views, output allocation, the stream lookup and a ctypes call of a dozen arguments) took 12-21 us of
// host time, so that small layers ran at the host's pace. Each function here takes the usual call as it
// is: plain contiguous, 16-byte aligned tensors of the right types and shapes on the current device.
// Anything else returns None, and the Python form, which handles every other case and raises every
// error, runs instead. A negative QMM4_ERR_* code of the library is returned as an int.
//
// Nothing is kept between calls: every property is read from the tensors on each call. The GIL is
// released around the library's call, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/util/SmallVector.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>

#include "qmm4.h"
#include "qmm_general.h"

namespace {

decltype(&qmm4_affine_bf16) p_affine = nullptr;
decltype(&qmm4_gate_up_silu_bf16) p_gate_up = nullptr;
decltype(&qmm_affine_general_bf16) p_general = nullptr;
decltype(&qmm4_add_rms_norm_bf16) p_norm = nullptr;
decltype(&qmm4_add_rms_norm_qmm_bf16) p_norm_qmm = nullptr;

// A plain tensor on a HIP device, contiguous with data on an `align`-byte boundary, or null: no
// subclass, no wrapper of a transform or a mode, nothing whose storage is not its own.
const at::Tensor* plain(PyObject* o, size_t align) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided) return nullptr;
  const c10::DispatchKeySet ks = t.key_set();
  if (ks.has(c10::DispatchKey::Python) || ks.has(c10::DispatchKey::FuncTorchBatched) ||
      ks.has(c10::DispatchKey::FuncTorchGradWrapper) || ks.has(c10::DispatchKey::Functionalize) ||
      ks.has(c10::DispatchKey::Conjugate) || ks.has(c10::DispatchKey::Negative) || ks.has(c10::DispatchKey::Batched))
    return nullptr;
  if (!t.has_storage() || !t.is_contiguous() || t.numel() == 0) return nullptr;
  if (reinterpret_cast<uintptr_t>(t.const_data_ptr()) % align != 0) return nullptr;
  return &t;
}

bool same_current_device(const at::Tensor& x, std::initializer_list<const at::Tensor*> others) {
  const auto d = x.device();
  for (const at::Tensor* t : others)
    if (t->device() != d) return false;
  return d.index() == c10::hip::current_device() && !c10::impl::TorchDispatchModeTLS::any_modes_set();
}

void* stream_of(const at::Tensor& x) {
  return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(x.device().index()).stream();
}

void* ptr(const at::Tensor& t) { return const_cast<void*>(t.const_data_ptr()); }
// A new output's data, or null where a transform hands out a wrapper without storage of its own.
void* out_ptr(const at::Tensor& t) { return t.has_storage() && t.is_cuda() ? ptr(t) : nullptr; }

struct Weights {
  const uint32_t* w;
  const void *s, *b;
  Weights(const at::Tensor& codes, const at::Tensor& scales, const at::Tensor& biases)
      : w(static_cast<const uint32_t*>(ptr(codes))), s(ptr(scales)), b(ptr(biases)) {}
};

bool is_codes(const at::Tensor& w) { return w.dim() == 2 && (w.scalar_type() == at::kInt || w.scalar_type() == at::kUInt32); }
bool is_bf16(const at::Tensor& t) { return t.scalar_type() == at::kBFloat16; }

at::Tensor empty_like_rows(const at::Tensor& x, int64_t n) {
  c10::SmallVector<int64_t, 8> sizes(x.sizes().begin(), x.sizes().end());
  sizes.back() = n;
  return at::empty(sizes, x.options());
}

// w [n, k * bits / 32] with scales and biases [n, k / group] for x's last dimension k.
bool weights_match(const at::Tensor& w, const at::Tensor& s, const at::Tensor& b, int64_t k, int64_t group, int64_t bits) {
  return is_codes(w) && is_bf16(s) && is_bf16(b) && s.dim() == 2 && b.dim() == 2 && k % group == 0 &&
         w.size(1) * 32 == k * bits && s.size(0) == w.size(0) && b.size(0) == w.size(0) && s.size(1) == k / group &&
         b.size(1) == k / group;
}

// Whether something sees or rewrites torch's own operations (same_current_device declines for dispatch
// modes): the general path's library product is one of them, the kernel is not.
bool observed() {
  return at::impl::torch_function_mode_enabled() ||
         (at::autocast::is_autocast_enabled(at::kCUDA) && at::autocast::get_autocast_dtype(at::kCUDA) != at::kBFloat16);
}

PyObject* none() { Py_RETURN_NONE; }

// `expr` runs without the GIL: it touches no tensor and throws nothing (pointers are taken before).
#define CALL(rc, expr)   \
  Py_BEGIN_ALLOW_THREADS \
  rc = (expr);           \
  Py_END_ALLOW_THREADS

// qmm(x, w, scales, biases, group_size, bits, general): quantized_matmul of 4-bit groups of 64 on the
// packed kernels, or of any format on the general kernel when `general` is true (the caller's rule).
PyObject* qmm(PyObject*, PyObject* const* a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 7) return none();
  const at::Tensor *x = plain(a[0], 16), *w = plain(a[1], 16), *s = plain(a[2], 16), *b = plain(a[3], 16);
  if (!x || !w || !s || !b || !is_bf16(*x) || x->dim() < 1 || !same_current_device(*x, {w, s, b})) return none();
  const int64_t group = PyLong_AsLongLong(a[4]), bits = PyLong_AsLongLong(a[5]);
  if (PyErr_Occurred()) return nullptr;
  const bool general = a[6] == Py_True;
  const int64_t k = x->sizes().back(), m = x->numel() / k, n = w->size(0);
  if (group <= 0 || bits <= 0 || !weights_match(*w, *s, *b, k, group, bits) || (general && observed())) return none();
  at::Tensor y = empty_like_rows(*x, n);
  const Weights q(*w, *s, *b);
  void *st = stream_of(*x), *xp = ptr(*x), *yp = out_ptr(y);
  if (!yp) return none();
  int rc;
  if (general) {
    CALL(rc, p_general(xp, q.w, q.s, q.b, yp, m, n, k, (int)group, (int)bits, st))
  } else {
    CALL(rc, p_affine(xp, q.w, q.s, q.b, yp, m, n, k, (int)group, (int)bits, 1, st))
  }
  return rc == 0 ? THPVariable_Wrap(std::move(y)) : PyLong_FromLong(rc);
  END_HANDLE_TH_ERRORS
}

// linear(x, w, scales, biases, w_ptr, scales_ptr, biases_ptr): a bound 4-bit layer; None as well when a
// tensor's data no longer lies where it was bound (the caller rebinds).
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 7) return none();
  const at::Tensor *x = plain(a[0], 16), *w = plain(a[1], 16), *s = plain(a[2], 16), *b = plain(a[3], 16);
  if (!x || !w || !s || !b || !is_bf16(*x) || x->dim() < 1 || !same_current_device(*x, {w, s, b})) return none();
  if (ptr(*w) != PyLong_AsVoidPtr(a[4]) || ptr(*s) != PyLong_AsVoidPtr(a[5]) || ptr(*b) != PyLong_AsVoidPtr(a[6]))
    return PyErr_Occurred() ? nullptr : none();
  const int64_t k = x->sizes().back(), m = x->numel() / k, n = w->size(0);
  if (!weights_match(*w, *s, *b, k, 64, 4)) return none();
  at::Tensor y = empty_like_rows(*x, n);
  const Weights q(*w, *s, *b);
  void *st = stream_of(*x), *xp = ptr(*x), *yp = out_ptr(y);
  if (!yp) return none();
  int rc;
  CALL(rc, p_affine(xp, q.w, q.s, q.b, yp, m, n, k, 64, 4, 1, st))
  return rc == 0 ? THPVariable_Wrap(std::move(y)) : PyLong_FromLong(rc);
  END_HANDLE_TH_ERRORS
}

// gate_up(x, w, scales, biases): gate_up_silu of 4-bit groups of 64.
PyObject* gate_up(PyObject*, PyObject* const* a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 4) return none();
  const at::Tensor *x = plain(a[0], 16), *w = plain(a[1], 16), *s = plain(a[2], 16), *b = plain(a[3], 16);
  if (!x || !w || !s || !b || !is_bf16(*x) || x->dim() < 1 || !same_current_device(*x, {w, s, b})) return none();
  const int64_t k = x->sizes().back(), m = x->numel() / k, n = w->size(0);
  if (n % 32 != 0 || !weights_match(*w, *s, *b, k, 64, 4)) return none();
  at::Tensor y = empty_like_rows(*x, n / 2);
  const Weights q(*w, *s, *b);
  void *st = stream_of(*x), *xp = ptr(*x), *yp = out_ptr(y);
  if (!yp) return none();
  int rc;
  CALL(rc, p_gate_up(xp, q.w, q.s, q.b, yp, m, n, k, 64, 4, 1, st))
  return rc == 0 ? THPVariable_Wrap(std::move(y)) : PyLong_FromLong(rc);
  END_HANDLE_TH_ERRORS
}

// x, r and the norm weight of add_rms_norm: bf16, x and r of one shape, weight of its last dimension.
bool norm_args(const at::Tensor* x, const at::Tensor* r, const at::Tensor* w) {
  return x && r && w && is_bf16(*x) && is_bf16(*r) && is_bf16(*w) && x->dim() >= 1 && x->sizes() == r->sizes() &&
         w->dim() == 1 && w->size(0) == x->sizes().back();
}

// norm(x, r, weight, eps): (h, n) of add_rms_norm.
PyObject* norm(PyObject*, PyObject* const* a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 4 || !PyFloat_Check(a[3])) return none();
  const at::Tensor *x = plain(a[0], 16), *r = plain(a[1], 16), *w = plain(a[2], 16);
  if (!norm_args(x, r, w) || !same_current_device(*x, {r, w})) return none();
  const int64_t d = x->sizes().back(), m = x->numel() / d;
  at::Tensor h = at::empty(x->sizes(), x->options()), n = at::empty(x->sizes(), x->options());
  void *st = stream_of(*x), *xp = ptr(*x), *rp = ptr(*r), *wp = ptr(*w), *hp = out_ptr(h), *np = out_ptr(n);
  if (!hp || !np) return none();
  const float eps = (float)PyFloat_AS_DOUBLE(a[3]);
  int rc;
  CALL(rc, p_norm(xp, rp, wp, hp, np, m, d, eps, st))
  if (rc != 0) return PyLong_FromLong(rc);
  PyObject* out = PyTuple_New(2);
  if (!out) return nullptr;
  PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(h)));
  PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(n)));
  return out;
  END_HANDLE_TH_ERRORS
}

// norm_qmm(x, r, weight, eps, w, scales, biases, silu_mul): (h, n, y) of add_rms_norm_qmm_.
PyObject* norm_qmm(PyObject*, PyObject* const* a, Py_ssize_t na) {
  HANDLE_TH_ERRORS
  if (na != 8 || !PyFloat_Check(a[3])) return none();
  const at::Tensor *x = plain(a[0], 16), *r = plain(a[1], 16), *nw = plain(a[2], 16), *w = plain(a[4], 16),
                   *s = plain(a[5], 16), *b = plain(a[6], 16);
  if (!norm_args(x, r, nw) || !w || !s || !b || !same_current_device(*x, {r, nw, w, s, b})) return none();
  const bool silu = a[7] == Py_True;
  const int64_t k = x->sizes().back(), m = x->numel() / k, n = w->size(0);
  if ((silu && n % 32 != 0) || !weights_match(*w, *s, *b, k, 64, 4)) return none();
  at::Tensor h = at::empty(x->sizes(), x->options()), nn = at::empty(x->sizes(), x->options());
  at::Tensor y = empty_like_rows(*x, silu ? n / 2 : n);
  const Weights q(*w, *s, *b);
  void *st = stream_of(*x), *xp = ptr(*x), *rp = ptr(*r), *np = ptr(*nw);
  void *hp = out_ptr(h), *nnp = out_ptr(nn), *yp = out_ptr(y);
  if (!hp || !nnp || !yp) return none();
  const float eps = (float)PyFloat_AS_DOUBLE(a[3]);
  int rc;
  CALL(rc, p_norm_qmm(xp, rp, np, eps, hp, nnp, q.w, q.s, q.b, yp, m, n, k, 64, 4, 1,
                      silu ? QMM4_EPILOGUE_SILU_MUL : QMM4_EPILOGUE_NONE, st))
  if (rc != 0) return PyLong_FromLong(rc);
  PyObject* out = PyTuple_New(3);
  if (!out) return nullptr;
  PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(h)));
  PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(nn)));
  PyTuple_SET_ITEM(out, 2, THPVariable_Wrap(std::move(y)));
  return out;
  END_HANDLE_TH_ERRORS
}

// bind(affine, gate_up, general, norm, norm_qmm): the addresses of the loaded library's functions.
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t na) {
  if (na != 5) {
    PyErr_SetString(PyExc_TypeError, "bind takes 5 addresses");
    return nullptr;
  }
  void* p[5];
  for (int i = 0; i < 5; ++i) {
    p[i] = PyLong_AsVoidPtr(a[i]);
    if (!p[i]) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null function address");
      return nullptr;
    }
  }
  p_affine = reinterpret_cast<decltype(p_affine)>(p[0]);
  p_gate_up = reinterpret_cast<decltype(p_gate_up)>(p[1]);
  p_general = reinterpret_cast<decltype(p_general)>(p[2]);
  p_norm = reinterpret_cast<decltype(p_norm)>(p[3]);
  p_norm_qmm = reinterpret_cast<decltype(p_norm_qmm)>(p[4]);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&bind)), METH_FASTCALL, nullptr},
    {"qmm", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&qmm)), METH_FASTCALL, nullptr},
    {"linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&linear)), METH_FASTCALL, nullptr},
    {"gate_up", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&gate_up)), METH_FASTCALL, nullptr},
    {"norm", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&norm)), METH_FASTCALL, nullptr},
    {"norm_qmm", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&norm_qmm)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) {
  PyObject* m = PyModule_Create(&module);
  // The torch this was built for (the loader refuses another: ATen's layouts are not stable).
  if (m && PyModule_AddStringConstant(m, "TORCH_VERSION", QMM4_TORCH_VERSION) < 0) Py_CLEAR(m);
  return m;
}
