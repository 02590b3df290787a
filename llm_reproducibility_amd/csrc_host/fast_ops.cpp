// The common calls of the row-wise operators (RMSNorm with and without residual, SiLU * up, mean, log_softmax) without
// Python between the tensors and the launch.  A call on a few rows is host time: checks, two output allocations and thirteen
// arguments marshalled one by one took 9.6 us around a kernel of 3 (add-RMSNorm of 7 rows), here 4.
//
// Every function takes the plain case only (ordinary dense tensors of one type on the current device, rows that
// the kernels read as they are) and returns None for everything else, refusals and errors of the library included: the
// caller then goes the long way in ops.py, which converts, copies or raises.  Nothing is kept between calls.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/tbik_hip.h"

namespace {

// a plain dense tensor on the current device (neither a subclass nor a lazy or nested one)
bool plain(PyObject* o, int dev) {
  if (!THPVariable_CheckExact(o)) return false;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.layout() == at::kStrided && t.is_cuda() && t.get_device() == dev && !t.is_neg() && !t.is_conj();
}

struct Rows {
  const void* p;
  int64_t rows, cols, ld;
};
// a 16-bit matrix whose rows the kernels read in place: contiguous columns, 16-byte aligned rows
bool rows16(const at::Tensor& t, Rows* r) {
  if (t.dim() != 2) return false;
  *r = Rows{t.data_ptr(), t.size(0), t.size(1), t.size(0) == 1 ? t.size(1) : t.stride(0)};
  return r->rows > 0 && r->cols > 0 && r->cols % 8 == 0 && t.stride(1) == 1 && r->ld >= r->cols && r->ld % 8 == 0 &&
         (reinterpret_cast<uintptr_t>(r->p) & 15) == 0;
}
bool vec16(const at::Tensor& t, const at::Tensor& like, int64_t n) {
  return t.dim() == 1 && t.size(0) == n && (n == 1 || t.stride(0) == 1) && t.scalar_type() == like.scalar_type();
}
bool half(const at::Tensor& t) { return t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kHalf; }
int code(const at::Tensor& t) {
  return t.scalar_type() == at::kFloat ? 0 : t.scalar_type() == at::kBFloat16 ? 1 : t.scalar_type() == at::kHalf ? 2 : -1;
}
// a flag that is Python's own bool; whatever else counts as true or false there (0, 1, a numpy bool) goes the long way
bool flag(PyObject* o, bool* v) {
  *v = o == Py_True;
  return PyBool_Check(o);
}
void* stream_of(int dev) { return static_cast<void*>(c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(dev)).stream()); }

// the launch, other Python threads free to run meanwhile (it may wait for room in the queue)
template <typename F>
int launch(F&& f) {
  PyThreadState* save = PyEval_SaveThread();
  const int rc = f();
  PyEval_RestoreThread(save);
  return rc;
}

// f() gives the result or an undefined tensor (None); a C++ exception is left to the long way as well, which meets its cause
template <typename F>
PyObject* or_none(F&& f) {
  try {
    at::Tensor t = f(static_cast<int>(c10::hip::current_device()));
    if (t.defined()) return THPVariable_Wrap(std::move(t));
  } catch (const std::exception&) {
  }
  PyErr_Clear();
  Py_RETURN_NONE;
}

// rms_norm(x, weight or None, eps)
PyObject* rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 3 || !PyFloat_CheckExact(a[2])) Py_RETURN_NONE;
  return or_none([&](int dev) -> at::Tensor {
    Rows x;
    if (!plain(a[0], dev)) return {};
    const at::Tensor& t = THPVariable_Unpack(a[0]);
    if (!half(t) || !rows16(t, &x) || x.cols > INT32_MAX) return {};
    const void* w = nullptr;
    if (a[1] != Py_None) {
      if (!plain(a[1], dev) || !vec16(THPVariable_Unpack(a[1]), t, x.cols)) return {};
      w = THPVariable_Unpack(a[1]).data_ptr();
    }
    at::Tensor out = at::empty({x.rows, x.cols}, t.options());
    const auto fn = t.scalar_type() == at::kHalf ? bi_rmsnorm_f16 : bi_rmsnorm_bf16;
    const float eps = static_cast<float>(PyFloat_AS_DOUBLE(a[2]));
    void *o = out.data_ptr(), *st = stream_of(dev);
    const int rc = launch([&] { return fn(x.p, x.ld, nullptr, 0, w, o, x.cols, nullptr, 0, x.rows, static_cast<int>(x.cols), eps, st); });
    return rc == TBIK_OK ? out : at::Tensor();
  });
}

// add_rms_norm(x, residual, weight or None, eps) -> [normalised, sum]
PyObject* add_rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 4 || !PyFloat_CheckExact(a[3])) Py_RETURN_NONE;
  at::Tensor sum;
  PyObject* out = or_none([&](int dev) -> at::Tensor {
    Rows x, r;
    if (!plain(a[0], dev) || !plain(a[1], dev)) return {};
    const at::Tensor &t = THPVariable_Unpack(a[0]), &res = THPVariable_Unpack(a[1]);
    if (!half(t) || res.scalar_type() != t.scalar_type() || !rows16(t, &x) || !rows16(res, &r) || x.cols > INT32_MAX) return {};
    if (r.rows != x.rows || r.cols != x.cols) return {};
    const void* w = nullptr;
    if (a[2] != Py_None) {
      if (!plain(a[2], dev) || !vec16(THPVariable_Unpack(a[2]), t, x.cols)) return {};
      w = THPVariable_Unpack(a[2]).data_ptr();
    }
    at::Tensor o = at::empty({x.rows, x.cols}, t.options());
    at::Tensor s = at::empty({x.rows, x.cols}, t.options());
    const auto fn = t.scalar_type() == at::kHalf ? bi_rmsnorm_f16 : bi_rmsnorm_bf16;
    const float eps = static_cast<float>(PyFloat_AS_DOUBLE(a[3]));
    void *op = o.data_ptr(), *sp = s.data_ptr(), *st = stream_of(dev);
    const int rc = launch([&] { return fn(x.p, x.ld, r.p, r.ld, w, op, x.cols, sp, x.cols, x.rows, static_cast<int>(x.cols), eps, st); });
    if (rc != TBIK_OK) return {};
    sum = std::move(s);
    return o;
  });
  if (!out || out == Py_None) return out;
  PyObject* list = PyList_New(2);
  PyObject* s = list ? THPVariable_Wrap(std::move(sum)) : nullptr;
  if (!s) {
    Py_DECREF(out);
    Py_XDECREF(list);
    return nullptr;
  }
  PyList_SET_ITEM(list, 0, out);
  PyList_SET_ITEM(list, 1, s);
  return list;
}

// silu_mul(gate_up)
PyObject* silu_mul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 1) Py_RETURN_NONE;
  return or_none([&](int dev) -> at::Tensor {
    Rows x;
    if (!plain(a[0], dev)) return {};
    const at::Tensor& t = THPVariable_Unpack(a[0]);
    if (!half(t) || !rows16(t, &x) || x.cols % 16 != 0 || x.cols > INT32_MAX) return {};
    const int64_t inter = x.cols / 2;
    at::Tensor out = at::empty({x.rows, inter}, t.options());
    const auto fn = t.scalar_type() == at::kHalf ? bi_silu_mul_f16 : bi_silu_mul_bf16;
    void *o = out.data_ptr(), *st = stream_of(dev);
    const int rc = launch([&] { return fn(x.p, x.ld, o, inter, x.rows, static_cast<int>(inter), st); });
    return rc == TBIK_OK ? out : at::Tensor();
  });
}

// mean_last(x, keepdim): the mean over the last dimension of a contiguous tensor
PyObject* mean_last(PyObject*, PyObject* const* a, Py_ssize_t n) {
  bool keepdim;
  if (n != 2 || !flag(a[1], &keepdim)) Py_RETURN_NONE;
  return or_none([&](int dev) -> at::Tensor {
    if (!plain(a[0], dev)) return {};
    const at::Tensor& t = THPVariable_Unpack(a[0]);
    if (t.dim() < 1 || !t.is_contiguous() || t.numel() == 0 || code(t) < 0) return {};
    const int64_t cols = t.size(-1), rows = t.numel() / cols;
    c10::SmallVector<int64_t, 6> shape(t.sizes().begin(), t.sizes().end() - 1);
    if (keepdim) shape.push_back(1);
    at::Tensor out = at::empty(shape, t.options());
    void *o = out.data_ptr(), *st = stream_of(dev);
    const void* in = t.data_ptr();
    const int rc = launch([&] { return bi_mean_dim(in, o, rows, cols, 1, code(t), st); });
    return rc == TBIK_OK ? out : at::Tensor();
  });
}

// log_softmax(x, write_softmax, to_float) over the rows of a matrix
PyObject* log_softmax(PyObject*, PyObject* const* a, Py_ssize_t n) {
  bool soft, to_float;
  if (n != 3 || !flag(a[1], &soft) || !flag(a[2], &to_float)) Py_RETURN_NONE;
  return or_none([&](int dev) -> at::Tensor {
    if (!plain(a[0], dev)) return {};
    const at::Tensor& t = THPVariable_Unpack(a[0]);
    if (t.dim() != 2 || t.numel() == 0 || code(t) < 0 || t.stride(1) != 1 || (t.size(0) > 1 && t.stride(0) < t.size(1))) return {};
    const int64_t rows = t.size(0), cols = t.size(1);
    at::Tensor out = at::empty({rows, cols}, to_float ? t.options().dtype(at::kFloat) : t.options());
    const size_t need = bi_log_softmax_workspace_bytes(rows, cols);
    at::Tensor ws;
    if (need) ws = at::empty({static_cast<int64_t>((need + 3) / 4)}, t.options().dtype(at::kFloat));
    void *o = out.data_ptr(), *st = stream_of(dev), *wp = need ? ws.data_ptr() : nullptr;
    const void* in = t.data_ptr();
    const int rc = launch([&] { return bi_log_softmax(in, rows > 1 ? t.stride(0) : cols, code(t), o, cols, code(out), rows, cols, wp, need, soft, st); });
    return rc == TBIK_OK ? out : at::Tensor();
  });
}

#define FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST(rms_norm), FAST(add_rms_norm), FAST(silu_mul), FAST(mean_last), FAST(log_softmax), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fast", "common calls of the row-wise operators", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// built_for (TBIK_BUILT_FOR, from build.py): the library's ABI and the torch this was compiled against; ops.py compares it with what
// it runs with before the first call
PyMODINIT_FUNC PyInit__fast(void) {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "built_for", TBIK_BUILT_FOR) != 0) Py_CLEAR(m);
  return m;
}
