// host_common.h — what the extension modules share: argument readers that decline (NotOrdinary) whatever is not the
// ordinary case, the interpreter's lock, a call's device and stream.  The reasons stand in host.cpp.
#pragma once
#include <Python.h>

#include <torch/csrc/autograd/python_variable.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include "../../include/triton_int_hip.h"

namespace {

using at::ScalarType;
using at::Tensor;

// Releases the interpreter's lock for its lifetime.
struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

struct NotOrdinary {};  // thrown by the argument readers, turned into None

void need(bool ok) {
  if (!ok) throw NotOrdinary{};
}

// A call's device and stream: those of its first tensor, which has to be on the current device.
struct Call {
  c10::DeviceIndex dev;
  void* stream;
  explicit Call(const Tensor& t) : dev(t.get_device()) {
    need(dev == c10::hip::current_device());
    stream = (void*)c10::hip::getCurrentHIPStream(dev).stream();
  }
  Tensor empty(at::IntArrayRef sizes, ScalarType type) const {
    return Tensor(at::detail::empty_cuda(sizes, type, c10::Device(c10::kCUDA, dev), std::nullopt));
  }
};

// A plain tensor on a GPU; `dev` < 0: on any.
const Tensor& tensor(PyObject* o, int dev = -1) {
  need(THPVariable_CheckExact(o));
  const Tensor& t = THPVariable_Unpack(o);
  need(t.is_cuda() && (dev < 0 || t.get_device() == dev));
  return t;
}

const Tensor& tensor(PyObject* o, int dev, ScalarType type) {
  const Tensor& t = tensor(o, dev);
  need(t.scalar_type() == type);
  return t;
}

const void* ptr(const Tensor& t) { return t.const_data_ptr(); }
void* mptr(const Tensor& t) { return t.mutable_data_ptr(); }

// an optional contiguous vector of `n` elements of `type`
const void* vector(PyObject* o, int dev, ScalarType type, int64_t n) {
  if (o == Py_None) return nullptr;
  const Tensor& t = tensor(o, dev, type);
  need(t.numel() == n && t.is_contiguous());
  return ptr(t);
}

const float* scale(PyObject* o, int dev) {
  if (o == Py_None) return nullptr;
  return (const float*)ptr(tensor(o, dev, ScalarType::Float));
}

int64_t integer(PyObject* o) {
  const int64_t v = PyLong_AsLongLong(o);
  need(!(v == -1 && PyErr_Occurred()));
  return v;
}

double number(PyObject* o) {
  need(PyFloat_Check(o) || PyLong_Check(o));
  const double v = PyFloat_AsDouble(o);
  need(!(v == -1.0 && PyErr_Occurred()));  // an integer beyond any double
  return v;
}

// A Python bool itself: anything else that counts as true or false is for the Python path to convert.
bool flag(PyObject* o) {
  need(PyBool_Check(o));
  return o == Py_True;
}

int bias_kind(ScalarType t) {
  switch (t) {
    case ScalarType::Char: return TI_BIAS_I8;
    case ScalarType::Int: return TI_BIAS_I32;
    case ScalarType::Float: return TI_BIAS_F32;
    case ScalarType::Half: return TI_BIAS_F16;
    case ScalarType::BFloat16: return TI_BIAS_BF16;
    default: throw NotOrdinary{};
  }
}

ScalarType out_type(int dt) {
  switch (dt) {
    case TI_I8: return ScalarType::Char;
    case TI_I32: return ScalarType::Int;
    case TI_F32: return ScalarType::Float;
    case TI_F16: return ScalarType::Half;
    case TI_BF16: return ScalarType::BFloat16;
    default: throw NotOrdinary{};
  }
}

int dtype_code(ScalarType t) {
  switch (t) {
    case ScalarType::Float: return TI_F32;
    case ScalarType::Half: return TI_F16;
    case ScalarType::BFloat16: return TI_BF16;
    default: throw NotOrdinary{};
  }
}

int int32_size(int64_t v) {
  need(v >= 0 && v <= 0x7fffffff);
  return (int)v;
}

// Distance of the rows [..., n] with unit stride along the last dimension and one distance between all of them (a
// slice of wider rows); n for a single row.  Anything else needs a copy.
int64_t row_pitch(const Tensor& t) {
  const int64_t d = t.dim();
  need(d >= 1);
  int64_t pitch = t.size(d - 1), next = -1;
  if (t.is_contiguous()) return pitch;
  need(t.stride(d - 1) == 1);
  for (int64_t i = d - 2; i >= 0; --i) {
    if (t.size(i) == 1) continue;
    if (next < 0) pitch = t.stride(i);
    need(next < 0 || t.stride(i) == next);
    next = t.stride(i) * t.size(i);
  }
  return pitch;
}

// activations [..., K] as M rows of one pitch
struct Rows {
  int M, K;
  int64_t pitch;
  Rows(const Tensor& a, int64_t k) {
    need(a.dim() >= 2 && a.size(-1) == k && k > 0);
    K = int32_size(k);
    M = int32_size(a.numel() / k);
    pitch = row_pitch(a);
  }
};

c10::SmallVector<int64_t, 6> with_last(const Tensor& a, int64_t n) {
  c10::SmallVector<int64_t, 6> s(a.sizes().begin(), a.sizes().end());
  s.back() = n;
  return s;
}

template <class F>
PyObject* guarded(Py_ssize_t n, Py_ssize_t want, F f) {
  if (n != want) {
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
    return nullptr;
  }
  try {
    return f();
  } catch (const NotOrdinary&) {
  } catch (const std::exception&) {  // nothing is launched yet: the allocations come first
  }
  PyErr_Clear();
  Py_RETURN_NONE;
}

// A K cache [seqs*heads, T, D] and a V^T cache [seqs*heads, D, T]: addresses of the last S positions
struct Caches {
  int64_t BH, T, D;
  int8_t *k = nullptr, *vt;
  int64_t k_hs = 0, k_rs = 0, vt_rs;
  Caches(PyObject* ko, PyObject* vo, int dev, int64_t S) {
    const Tensor& v = tensor(vo, dev, ScalarType::Char);
    need(v.dim() == 3);
    BH = v.size(0), D = v.size(1), T = v.size(2);
    need(D % 16 == 0 && S <= T && (v.stride(2) == 1 || T == 1) && (v.stride(0) == D * v.stride(1) || BH == 1));
    vt_rs = v.stride(1);
    vt = (int8_t*)mptr(v) + (T - S);
    if (ko == Py_None) return;
    const Tensor& kc = tensor(ko, dev, ScalarType::Char);
    need(kc.dim() == 3 && kc.size(0) == BH && kc.size(1) == T && kc.size(2) == D && kc.stride(2) == 1);
    k_hs = kc.stride(0), k_rs = kc.stride(1);
    k = (int8_t*)mptr(kc) + (T - S) * k_rs;
  }
};

}  // namespace
