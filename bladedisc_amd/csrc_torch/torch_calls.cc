// The host side of bladedisc_amd/kernels.py: takes torch tensors, fills in sizes, strides, the
// result and the scratch, and calls the C ABI of include/disc_q8.h on the current stream.
//
// What bounds it: nothing but instructions on the calling thread.  A quantized linear of a small
// batch runs 3-5 us on the GPU; driven through ctypes (one Python object per argument, a stream
// object, three reshapes of one-element scales, two library calls for the scratch) the call
// itself took 12-14 us and the GPU waited for it.  Here a call costs the launch plus about a
// microsecond.  Results and scratch come from torch's caching allocator on the current stream,
// as torch.empty does, so nothing outlives the call and streams and threads behave as before;
// the interpreter lock is released around the launch.
#define PY_SSIZE_T_CLEAN
#include <torch/csrc/python_headers.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>

#include "disc_q8.h"
#include "status_words.h"
#include "unlocked.h"

namespace {

using at::ScalarType;
using at::Tensor;

struct PyFailure {};   // a Python exception has been set

[[noreturn]] void raise(PyObject* type, const char* msg) {
  PyErr_SetString(type, msg);
  throw PyFailure{};
}

void check(int status, const char* what) {
  if (status == 0) return;
  PyErr_Format(PyExc_RuntimeError, "%s failed: %s", what, dq8_last_error());
  throw PyFailure{};
}

void* stream() { return (void*)c10::hip::getCurrentHIPStream().stream(); }

// The launch itself, without the interpreter lock: f(args...), the arguments read before.
template <typename... P, typename... A>
void launch(const char* what, int (*f)(P...), A... args) {
  check(dq8::call_unlocked(f, args...), what);
}

Tensor empty(at::IntArrayRef sizes, ScalarType t, const at::Device& dev) {
  return Tensor(at::detail::empty_cuda(sizes, t, dev, std::nullopt));
}

const Tensor& tensor(PyObject* o) {
  if (!THPVariable_Check(o)) raise(PyExc_TypeError, "expected a tensor");
  return THPVariable_Unpack(o);
}

const Tensor& device_tensor(PyObject* o) {
  const Tensor& t = tensor(o);
  if (!t.is_cuda()) raise(PyExc_ValueError, "expected device tensors");
  return t;
}

// None or a device tensor
Tensor optional_device_tensor(PyObject* o) {
  return o == Py_None ? Tensor() : device_tensor(o);
}

// what is read, and what is written (a lazy copy becomes a real one first)
const void* in(const Tensor& t) { return t.defined() ? t.const_data_ptr() : nullptr; }
void* inout(const Tensor& t) { return t.defined() ? t.mutable_data_ptr() : nullptr; }

int64_t integer(PyObject* o) {
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw PyFailure{};
  return v;
}

// int(o): a float as well
int64_t as_integer(PyObject* o) {
  if (PyLong_Check(o)) return integer(o);
  PyObject* made = PyNumber_Long(o);
  if (!made) throw PyFailure{};
  const int64_t v = PyLong_AsLongLong(made);
  Py_DECREF(made);
  if (v == -1 && PyErr_Occurred()) throw PyFailure{};
  return v;
}

bool truth(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw PyFailure{};
  return v != 0;
}

Tensor dense(const Tensor& t) { return t.is_contiguous() ? t : t.contiguous(); }

// A scale operand: a flat f32 device tensor, a number, or a sequence or array of numbers.
Tensor scale(PyObject* o, const at::Device& dev) {
  if (o == Py_None) return Tensor();
  if (THPVariable_Check(o)) {
    const Tensor& t = THPVariable_Unpack(o);
    if (t.scalar_type() == ScalarType::Float && t.is_contiguous()) return t;
    return t.reshape({-1}).contiguous().to(ScalarType::Float);
  }
  if (PyFloat_Check(o) || (PyNumber_Check(o) && !PyObject_HasAttrString(o, "__len__"))) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw PyFailure{};
    return at::full({1}, v, at::TensorOptions().dtype(ScalarType::Float).device(dev));
  }
  // whatever else torch.tensor takes: lists, tuples, numpy arrays
  PyObject* mod = PyImport_ImportModule("torch");
  PyObject* made = mod ? PyObject_CallMethod(mod, "tensor", "(O)", o) : nullptr;
  Py_XDECREF(mod);
  if (!made) throw PyFailure{};
  const Tensor t = THPVariable_Unpack(made);
  Py_DECREF(made);
  return t.reshape({-1}).to(ScalarType::Float).to(dev).contiguous();
}

int64_t count(const Tensor& t) { return t.defined() ? t.numel() : 0; }

ScalarType epilogue_type(int64_t epilogue) {
  switch (epilogue) {
    case DQ8_EPI_ACC_S32: return ScalarType::Int;
    case DQ8_EPI_REQUANT_CPU:
    case DQ8_EPI_REQUANT_GPU:
    case DQ8_EPI_REQUANT_FIXEDPOINT: return ScalarType::Char;
    case DQ8_EPI_DEQUANT_F32:
    case DQ8_EPI_REQUANT_CPU_DEQUANT_F32:
    case DQ8_EPI_REQUANT_GPU_DEQUANT_F32: return ScalarType::Float;
  }
  raise(PyExc_KeyError, "unknown epilogue");
}

int bias_kind(const Tensor& b) {
  if (!b.defined()) return DQ8_BIAS_NONE;
  switch (b.scalar_type()) {
    case ScalarType::Int: return DQ8_BIAS_S32;
    case ScalarType::Float: return DQ8_BIAS_F32;
    case ScalarType::Char: return DQ8_BIAS_S8;
    default: raise(PyExc_KeyError, "bias type");
  }
}

// [outer, channels, inner] of a shape along an axis (None: one channel)
struct View3 {
  int64_t outer = 1, nch = 1, inner = 1;
  View3(const Tensor& x, PyObject* axis) {
    if (axis == Py_None) {
      inner = x.numel();
      return;
    }
    int64_t a = integer(axis);
    if (a < 0) a += x.dim();
    if (a < 0 || a >= x.dim()) raise(PyExc_IndexError, "axis out of range");
    for (int64_t i = 0; i < a; ++i) outer *= x.size(i);
    nch = x.size(a);
    for (int64_t i = a + 1; i < x.dim(); ++i) inner *= x.size(i);
  }
};

// The dq8_postops_t inside a ctypes structure (None: null); the buffer is held while in use.
struct Post {
  Py_buffer view{};
  const dq8_postops_t* p = nullptr;
  explicit Post(PyObject* o) {
    if (o == Py_None) return;
    if (PyObject_GetBuffer(o, &view, PyBUF_SIMPLE) != 0) throw PyFailure{};
    if (view.len != (Py_ssize_t)sizeof(dq8_postops_t)) raise(PyExc_TypeError, "expected a PostOps structure");
    p = static_cast<const dq8_postops_t*>(view.buf);
  }
  Post(const Post&) = delete;
  ~Post() {
    if (view.obj) PyBuffer_Release(&view);
  }
};

PyObject* wrap(PyObject* given, const Tensor& t) {
  if (given != Py_None) {
    Py_INCREF(given);
    return given;
  }
  return THPVariable_Wrap(t);
}

void arguments(const char* name, Py_ssize_t n, Py_ssize_t want) {
  if (n == want) return;
  PyErr_Format(PyExc_TypeError, "%s takes %zd arguments (%zd given)", name, want, n);
  throw PyFailure{};
}

template <typename F>
PyObject* guarded(F&& f) {
  HANDLE_TH_ERRORS
  try {
    return f();
  } catch (const PyFailure&) {
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

int float_kind(const Tensor& x, const char* refusal) {
  if (x.scalar_type() == ScalarType::Float) return DQ8_DTYPE_F32;
  if (x.scalar_type() == ScalarType::Half) return DQ8_DTYPE_F16;
  raise(PyExc_TypeError, refusal);
}

// quantize(x, scale, zero_point, axis, qmin, qmax, round_mode, kind, store_dtype, out)
PyObject* py_quantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    arguments("quantize", n, 10);
    const Tensor x = dense(device_tensor(a[0]));
    const Tensor &s = device_tensor(a[1]), &z = device_tensor(a[2]);
    const int xk = float_kind(x, "quantize takes f32 or f16 input");
    const View3 v(x, a[3]);
    const int64_t qmin = as_integer(a[4]), qmax = as_integer(a[5]);
    const int round_mode = (int)integer(a[6]), kind = (int)integer(a[7]);
    const Tensor out = a[9] != Py_None
                           ? tensor(a[9])
                           : empty(x.sizes(), reinterpret_cast<THPDtype*>(a[8])->scalar_type, x.device());
    const int64_t n_q = a[3] != Py_None ? s.numel() : 1;
    void* st = stream();
    launch("dq8_quantize", dq8_quantize_ex, in(x), xk, inout(out), kind, v.outer, v.nch, v.inner,
           (const float*)in(s), (const int32_t*)in(z), n_q, qmin, qmax, round_mode, st);
    return wrap(a[9], out);
  });
}

// dequantize(q, scale, zero_point, axis, kind, out)
PyObject* py_dequantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    arguments("dequantize", n, 6);
    const Tensor q = dense(device_tensor(a[0]));
    const Tensor &s = device_tensor(a[1]), &z = device_tensor(a[2]);
    const View3 v(q, a[3]);
    const int kind = (int)integer(a[4]);
    const Tensor out = a[5] != Py_None ? tensor(a[5]) : empty(q.sizes(), ScalarType::Float, q.device());
    const int64_t n_q = a[3] != Py_None ? s.numel() : 1;
    void* st = stream();
    launch("dq8_dequantize", dq8_dequantize_ex, in(q), kind, (float*)inout(out), v.outer, v.nch, v.inner,
           (const float*)in(s), (const int32_t*)in(z), n_q, st);
    return wrap(a[5], out);
  });
}

// fake_quant(x, scale, zero_point, axis, qmin, qmax, round_mode, out)
PyObject* py_fake_quant(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    arguments("fake_quant", n, 8);
    const Tensor &x0 = device_tensor(a[0]), &s = device_tensor(a[1]), &z = device_tensor(a[2]);
    if (x0.scalar_type() != ScalarType::Float) raise(PyExc_TypeError, "fake_quant takes float32 tensors");
    const Tensor x = dense(x0);
    const View3 v(x, a[3]);
    const int qmin = (int)integer(a[4]), qmax = (int)integer(a[5]), round_mode = (int)integer(a[6]);
    const Tensor out = a[7] != Py_None ? tensor(a[7]) : empty(x.sizes(), ScalarType::Float, x.device());
    const int64_t n_q = a[3] != Py_None ? s.numel() : 1;
    void* st = stream();
    launch("dq8_fake_quant", dq8_fake_quant, (const float*)in(x), (float*)inout(out), v.outer, v.nch,
           v.inner, (const float*)in(s), (const int32_t*)in(z), n_q, qmin, qmax, round_mode, st);
    return wrap(a[7], out);
  });
}

// minmax(x, min_io, max_io, axis, workspace)
PyObject* py_minmax(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    arguments("minmax", n, 5);
    const Tensor &x0 = device_tensor(a[0]), &lo = device_tensor(a[1]), &hi = device_tensor(a[2]);
    if (x0.scalar_type() != ScalarType::Float || lo.scalar_type() != ScalarType::Float ||
        hi.scalar_type() != ScalarType::Float)
      raise(PyExc_TypeError, "minmax takes float32 tensors");
    const Tensor x = dense(x0);
    const View3 v(x, a[3]);
    if (lo.numel() != v.nch || hi.numel() != v.nch) {
      PyErr_Format(PyExc_ValueError, "min / max state must have one entry per channel (%lld)",
                   (long long)v.nch);
      throw PyFailure{};
    }
    const size_t need = dq8_minmax_workspace_bytes(v.outer, v.nch, v.inner);
    Tensor ws;
    if (a[4] != Py_None) ws = tensor(a[4]);
    if (!ws.defined() || (size_t)ws.nbytes() < need)
      ws = empty({(int64_t)(need > 0 ? need : 1)}, ScalarType::Byte, x.device());
    void* st = stream();
    launch("dq8_minmax", dq8_minmax, (const float*)in(x), v.outer, v.nch, v.inner, (float*)inout(lo),
           (float*)inout(hi), inout(ws), ws.nbytes(), st);
    Py_RETURN_NONE;
  });
}

Tensor pinned_words(int64_t n) {
  return at::empty({n}, at::TensorOptions().dtype(ScalarType::Int).pinned_memory(true));
}

// (for the process: torch may be gone at its end)
dq8::StatusWords& status_words() {
  static constexpr int kWords = 64;
  static const Tensor* page = new Tensor(pinned_words(kWords * dq8::StatusWords::kStride));
  static dq8::StatusWords* words = new dq8::StatusWords(page->data_ptr<int32_t>(), kWords);
  return *words;
}

// observe(x, min_io, max_io, axis, symmetric, q_min, q_max, fake_quant)
//   -> (min <= max everywhere, scale, zero_point, fake-quantized x or None)
// One step of an observer: two to four kernels, the last of them with the fake quantization, and one
// wait for the answer whether the observed range is sound.
PyObject* py_observe(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    arguments("observe", n, 8);
    const Tensor &x0 = device_tensor(a[0]), &lo = device_tensor(a[1]), &hi = device_tensor(a[2]);
    if (x0.scalar_type() != ScalarType::Float || lo.scalar_type() != ScalarType::Float ||
        hi.scalar_type() != ScalarType::Float || !lo.is_contiguous() || !hi.is_contiguous())
      raise(PyExc_TypeError, "observe takes float32 tensors");
    const Tensor x = dense(x0);
    const View3 v(x, a[3]);
    if (lo.numel() != v.nch || hi.numel() != v.nch) {
      PyErr_Format(PyExc_ValueError, "min / max state must have one entry per channel (%lld)",
                   (long long)v.nch);
      throw PyFailure{};
    }
    const bool symmetric = truth(a[4]), fake = truth(a[7]);
    const int q_min = (int)integer(a[5]), q_max = (int)integer(a[6]);
    const size_t need = dq8_minmax_workspace_bytes(v.outer, v.nch, v.inner);
    const Tensor ws = empty({(int64_t)need}, ScalarType::Byte, x.device());
    const Tensor s = empty(lo.sizes(), ScalarType::Float, x.device());
    const Tensor z = empty(lo.sizes(), ScalarType::Int, x.device());
    Tensor y;
    if (fake) y = empty(x.sizes(), ScalarType::Float, x.device());
    const float* xp = (const float*)in(x);
    float *lop = (float*)inout(lo), *hip = (float*)inout(hi);
    float *sp = (float*)inout(s), *yp = (float*)inout(y);
    int32_t* zp = (int32_t*)inout(z);
    void* wsp = inout(ws);
    const c10::hip::HIPStream st = c10::hip::getCurrentHIPStream();
    void* raw = (void*)st.stream();
    dq8::StatusWord<Tensor> status(status_words(), [](Tensor* own) {
      *own = pinned_words(1);
      return own->data_ptr<int32_t>();
    });
    const char* what = fake ? "dq8_observe_fake_quant" : "dq8_observe";
    int failed;
    int32_t answer = 0;
    {
      const dq8::Unlocked unlocked;
      auto drain = [&] { st.synchronize(); };
      if (fake)
        failed = dq8_observe_fake_quant(xp, yp, v.outer, v.nch, v.inner, lop, hip, symmetric, q_min, q_max,
                                        sp, zp, status.hand_out(), wsp, need, raw);
      else
        failed = dq8_observe(xp, v.outer, v.nch, v.inner, lop, hip, symmetric, q_min, q_max,
                             sp, zp, status.hand_out(), wsp, need, raw);
      if (!failed) {
        answer = status.wait(drain);
      } else {
        try {
          status.settle(drain);
        } catch (...) {   // (the error of the launch is the one to report)
        }
      }
    }
    check(failed, what);
    PyObject* r = PyTuple_New(4);
    if (!r) throw PyFailure{};
    PyTuple_SET_ITEM(r, 0, PyBool_FromLong(answer == 1));
    PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(s));
    PyTuple_SET_ITEM(r, 2, THPVariable_Wrap(z));
    if (fake) {
      PyTuple_SET_ITEM(r, 3, THPVariable_Wrap(y));
    } else {
      Py_INCREF(Py_None);
      PyTuple_SET_ITEM(r, 3, Py_None);
    }
    return r;
  });
}

// lut8(q, table, out)
PyObject* py_lut8(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    arguments("lut8", n, 3);
    const Tensor &q0 = device_tensor(a[0]), &table = device_tensor(a[1]);
    if (q0.element_size() != 1 || table.element_size() != 1 || table.numel() != 256)
      raise(PyExc_TypeError, "lut8 takes 8-bit tensors and a 256-entry table");
    const Tensor q = dense(q0);
    const Tensor out = a[2] != Py_None ? tensor(a[2]) : empty(q.sizes(), table.scalar_type(), q.device());
    void* st = stream();
    launch("dq8_lut8", dq8_lut8, in(q), inout(out), q.numel(), in(table), st);
    return wrap(a[2], out);
  });
}

// weight_only_qgemm(x, w, scale, zero_points, bias, tp_b, out, workspace)
PyObject* py_weight_only(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    arguments("weight_only_qgemm", n, 8);
    Tensor x = device_tensor(a[0]);
    Tensor w = device_tensor(a[1]);
    Tensor s = device_tensor(a[2]);
    Tensor zp = optional_device_tensor(a[3]), bias = optional_device_tensor(a[4]);
    const int xk = float_kind(x, "weight_only_qgemm takes f32 or f16 activations");
    const ScalarType xt = x.scalar_type();
    const bool w_signed = w.scalar_type() == ScalarType::Char;
    if ((!w_signed && w.scalar_type() != ScalarType::Byte) || w.dim() != 2)
      raise(PyExc_TypeError, "weight_only_qgemm takes a uint8 / int8 weight matrix");
    if (x.dim() != 2 || x.stride(1) != 1) x = x.reshape({-1, x.size(-1)}).contiguous();
    w = dense(w);
    const bool tp_b = truth(a[5]);
    const int64_t N = tp_b ? w.size(0) : w.size(1), K = tp_b ? w.size(1) : w.size(0), M = x.size(0);
    if (x.size(1) != K) raise(PyExc_ValueError, "contraction dimensions differ");
    auto as = [](const Tensor& t, ScalarType want) {
      return t.scalar_type() == want ? dense(t) : t.to(want).contiguous();
    };
    s = as(s, xt);
    if (bias.defined()) bias = as(bias, xt);
    if (zp.defined()) zp = as(zp, ScalarType::Int);
    const Tensor out = a[6] != Py_None ? tensor(a[6]) : empty({M, N}, xt, x.device());
    Tensor ws;
    if (THPVariable_Check(a[7])) {
      ws = THPVariable_Unpack(a[7]);
    } else if (truth(a[7])) {
      const size_t need = dq8_weight_only_qgemm_workspace_bytes_for(in(x), xk, x.stride(0), in(w), w.stride(0), tp_b,
                                                                    M, N, K);
      if (need) ws = empty({(int64_t)need}, ScalarType::Byte, x.device());
    }
    const size_t ws_bytes = ws.defined() ? ws.nbytes() : 0;
    void* st = stream();
    launch("dq8_weight_only_qgemm", dq8_weight_only_qgemm, in(x), xk, x.stride(0), in(w), w_signed,
           w.stride(0), tp_b, in(s), (const int32_t*)in(zp), in(bias), inout(out), out.stride(0), M, N, K,
           inout(ws), ws_bytes, st);
    return wrap(a[6], out);
  });
}

// An operand matrix whose rows may be strided but whose elements are dense.
Tensor matrix(const Tensor& t) { return t.dim() != 2 || t.stride(1) != 1 ? t.contiguous() : t; }

int64_t leading(const Tensor& t) { return std::max(t.stride(0), t.size(1)); }

// qgemm(a, w, epilogue, sx, sw, so, bias, tp_a, tp_b, zx, zw, zo, out, post)
PyObject* py_qgemm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    arguments("qgemm", n, 14);
    const Tensor x = matrix(device_tensor(a[0])), w = matrix(device_tensor(a[1]));
    const Tensor bias = optional_device_tensor(a[6]);
    if (x.dim() != 2 || w.dim() != 2) raise(PyExc_ValueError, "qgemm takes matrices");
    const int64_t epilogue = integer(a[2]);
    const bool tp_a = truth(a[7]), tp_b = truth(a[8]);
    const int64_t M = x.size(tp_a ? 1 : 0), K = x.size(tp_a ? 0 : 1);
    const int64_t N = w.size(tp_b ? 0 : 1);
    if (K != w.size(tp_b ? 1 : 0)) raise(PyExc_ValueError, "mismatch contraction dim");
    const int zx = (int)integer(a[9]), zw = (int)integer(a[10]), zo = (int)integer(a[11]);
    const at::Device dev = x.device();
    const Tensor out = a[12] != Py_None ? tensor(a[12]) : empty({M, N}, epilogue_type(epilogue), dev);
    const Tensor sx = scale(a[3], dev), sw = scale(a[4], dev), so = scale(a[5], dev);
    const int kind = bias_kind(bias);
    const Post post(a[13]);
    const size_t need = dq8_qgemm_workspace_bytes_zp(M, N, K, tp_a, tp_b, zx, zw);
    Tensor ws;
    if (need) ws = empty({(int64_t)need}, ScalarType::Byte, dev);
    void* st = stream();
    launch("dq8_qgemm", dq8_qgemm_fused, (const int8_t*)in(x), leading(x), (const int8_t*)in(w),
           leading(w), inout(out), M ? out.stride(0) : N, M, N, K, tp_a, tp_b, (int)epilogue, in(bias), kind,
           (const float*)in(sx), count(sx), (const float*)in(sw), count(sw), (const float*)in(so),
           count(so), zx, zw, zo, inout(ws), need, post.p, st);
    return wrap(a[12], out);
  });
}

// qlinear_f32(x, w, epilogue, sx, sw, so, bias, zo, round_mode, out)
PyObject* py_qlinear_f32(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    arguments("qlinear_f32", n, 10);
    Tensor x = device_tensor(a[0]);
    const Tensor w = matrix(device_tensor(a[1]));
    const Tensor bias = optional_device_tensor(a[6]);
    const int64_t epilogue = integer(a[2]);
    if (x.dim() != 2 || x.stride(1) != 1) x = x.reshape({-1, x.size(-1)}).contiguous();
    if (w.dim() != 2) raise(PyExc_ValueError, "qlinear_f32 takes a weight matrix");
    const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
    if (w.size(1) != K) raise(PyExc_ValueError, "mismatch contraction dim");
    const at::Device dev = x.device();
    const Tensor out = a[9] != Py_None ? tensor(a[9]) : empty({M, N}, epilogue_type(epilogue), dev);
    const Tensor sx = scale(a[3], dev), sw = scale(a[4], dev), so = scale(a[5], dev);
    const int kind = bias_kind(bias);
    const int zo = (int)integer(a[7]), round_mode = (int)integer(a[8]);
    void* st = stream();
    launch("dq8_qlinear_f32", dq8_qlinear_f32, (const float*)in(x), leading(x), (const int8_t*)in(w),
           leading(w), inout(out), M ? out.stride(0) : N, M, N, K, (int)epilogue, in(bias), kind,
           (const float*)in(sx), (const float*)in(sw), count(sw), (const float*)in(so), count(so), zo,
           round_mode, st);
    return wrap(a[9], out);
  });
}

template <typename T, int N>
struct Numbers {
  T v[N];
  explicit Numbers(PyObject* o) {
    PyObject* s = PySequence_Fast(o, "expected a sequence of integers");
    if (!s) throw PyFailure{};
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(s);
    bool bad = n > N;
    for (int i = 0; i < N; ++i) v[i] = 0;
    for (Py_ssize_t i = 0; i < n && !bad; ++i) {
      const int64_t x = PyLong_AsLongLong(PySequence_Fast_GET_ITEM(s, i));
      bad = x == -1 && PyErr_Occurred();
      v[i] = (T)x;
    }
    Py_DECREF(s);
    if (bad) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_IndexError, "too many values");
      throw PyFailure{};
    }
  }
};

// qconv2d(x, w, padding, metadata, out_shape, epilogue, sx, sw, so, bias, zo, out, workspace, post)
PyObject* py_qconv2d(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    arguments("qconv2d", n, 14);
    const Tensor x = dense(device_tensor(a[0])), w = dense(device_tensor(a[1]));
    const Tensor bias = optional_device_tensor(a[9]);
    if (x.dim() != 4 || w.dim() != 4) raise(PyExc_ValueError, "qconv2d takes tensors of rank 4");
    const Numbers<int32_t, 4> padding(a[2]);
    const Numbers<int32_t, 17> md(a[3]);
    const Numbers<int64_t, 4> os(a[4]);
    const int64_t epilogue = integer(a[5]);
    const at::Device dev = x.device();
    const Tensor out = a[11] != Py_None ? tensor(a[11])
                                        : empty(at::IntArrayRef(os.v, 4), epilogue_type(epilogue), dev);
    const Tensor sx = scale(a[6], dev), sw = scale(a[7], dev), so = scale(a[8], dev);
    const int kind = bias_kind(bias), zo = (int)integer(a[10]);
    const Post post(a[13]);
    const int64_t *is = x.sizes().data(), *ws_ = w.sizes().data();
    const size_t need = truth(a[12]) ? dq8_qconv2d_workspace_bytes_ex(is, ws_, os.v, md.v) : 0;
    Tensor ws;
    if (need) ws = empty({(int64_t)need}, ScalarType::Byte, dev);
    void* st = stream();
    launch("dq8_qconv2d", dq8_qconv2d_fused, (const int8_t*)in(x), is, (const int8_t*)in(w), ws_,
           padding.v, md.v, inout(out), os.v, (int)epilogue, in(bias), kind, (const float*)in(sx),
           (const float*)in(sw), count(sw), (const float*)in(so), zo, inout(ws), need, post.p, st);
    return wrap(a[11], out);
  });
}

// attention(qkv [.., seq, 3 heads 64], heads, scale or None, qkv_scale or None): int8 result with a scale, else
// f32; qkv is f32, or with a qkv_scale int8
PyObject* py_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    arguments("attention", n, 4);
    const Tensor x = dense(device_tensor(a[0]));
    const Tensor sx = scale(a[3], x.device());
    if (x.scalar_type() != (sx.defined() ? ScalarType::Char : ScalarType::Float) || x.dim() != 3)
      raise(PyExc_TypeError, "attention takes a float32 tensor of rank 3, or an int8 one and its scale");
    if (sx.defined() && (!sx.is_cuda() || sx.numel() != 1))
      raise(PyExc_ValueError, "attention takes one scale of its int8 input, on the device");
    const int64_t heads = integer(a[1]), h3 = x.size(2);
    if (heads <= 0 || h3 % (3 * heads) != 0) raise(PyExc_ValueError, "attention: heads do not divide the channels");
    const Tensor s = optional_device_tensor(a[2]);
    const Tensor out = empty({x.size(0), x.size(1), h3 / 3}, s.defined() ? ScalarType::Char : ScalarType::Float,
                             x.device());
    void* st = stream();
    float* y = s.defined() ? nullptr : (float*)inout(out);
    int8_t* y_q = s.defined() ? (int8_t*)inout(out) : nullptr;
    if (sx.defined())
      launch("dq8_attention_i8", dq8_attention_i8, (const int8_t*)in(x), (const float*)in(sx), x.size(0), x.size(1),
             heads, h3 / 3 / heads, y, y_q, (const float*)in(s), st);
    else
      launch("dq8_attention_f32", dq8_attention_f32, (const float*)in(x), x.size(0), x.size(1), heads,
             h3 / 3 / heads, y, y_q, (const float*)in(s), st);
    return THPVariable_Wrap(out);
  });
}

// layer_norm(x, gamma, beta, eps, scale or None): y, or (y, int8 of y) with a scale
PyObject* py_layer_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    arguments("layer_norm", n, 5);
    const Tensor x = dense(device_tensor(a[0]));
    const Tensor &g = device_tensor(a[1]), &b = device_tensor(a[2]);
    if (x.scalar_type() != ScalarType::Float || g.scalar_type() != ScalarType::Float ||
        b.scalar_type() != ScalarType::Float || x.dim() < 1 || !g.is_contiguous() || !b.is_contiguous() ||
        g.numel() != x.size(-1) || b.numel() != x.size(-1))
      raise(PyExc_TypeError, "layer_norm takes float32 tensors, weight and bias of the last dimension");
    const float eps = (float)PyFloat_AsDouble(a[3]);
    if (PyErr_Occurred()) throw PyFailure{};
    const Tensor s = optional_device_tensor(a[4]);
    const int64_t cols = x.size(-1), rows = cols ? x.numel() / cols : 0;
    const Tensor y = empty(x.sizes(), ScalarType::Float, x.device());
    Tensor q;
    if (s.defined()) q = empty(x.sizes(), ScalarType::Char, x.device());
    void* st = stream();
    launch("dq8_layernorm_f32", dq8_layernorm_f32, (const float*)in(x), rows, cols, (const float*)in(g),
           (const float*)in(b), eps, (float*)inout(y), (int8_t*)inout(q), (const float*)in(s), st);
    if (!s.defined()) return THPVariable_Wrap(y);
    PyObject* r = PyTuple_New(2);
    if (!r) throw PyFailure{};
    PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(y));
    PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(q));
    return r;
  });
}

// encoder_layer(h [batch, seq, hidden], heads, eps, operands): operands holds, for the merged
// projection, the attention output and the two feed-forward linears in turn, (int8 weights [N, K], f32
// bias, input scale, weight scales, output scale), then the activation table between the last two, the
// layer norms' weights and biases, and the zero point 0.  None where anything is of another form.
// What kernels.py's quantize, qgemm, attention and layer_norm do one after the other for a layer with
// everything fused that can be, the same eight launches: called one by one, with a view and a postops
// structure between most of them, they take 45 to 48 us of the host's time, which is more than the GPU
// needs below about 300 tokens.  A layer of hidden size 768: 48.1 -> 34.5 us at 1 x 19 tokens, 45.2 ->
// 40.0 at 11 x 20, the same from 6 x 90 on; the first pass of a process 197 -> 137.
PyObject* py_encoder_layer(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    arguments("encoder_layer", n, 4);
    const Tensor& h0 = device_tensor(a[0]);
    const int64_t heads = integer(a[1]);
    const float eps = (float)PyFloat_AsDouble(a[2]);
    if (PyErr_Occurred()) throw PyFailure{};
    constexpr int kLinears = 4, kEach = 5, kOperands = kLinears * kEach + 6;
    if (!PyTuple_Check(a[3]) || PyTuple_GET_SIZE(a[3]) != kOperands)
      raise(PyExc_TypeError, "encoder_layer takes a tuple of 26 operands");
    if (h0.scalar_type() != ScalarType::Float || h0.dim() != 3 || heads <= 0 || h0.size(2) != heads * 64) Py_RETURN_NONE;
    const int64_t batch = h0.size(0), seq = h0.size(1), hidden = h0.size(2), M = batch * seq;
    const at::Device dev = h0.device();
    const Tensor* t[kOperands];
    for (int i = 0; i < kOperands; ++i) {
      PyObject* o = PyTuple_GET_ITEM(a[3], i);
      if (!THPVariable_Check(o)) Py_RETURN_NONE;
      t[i] = &THPVariable_Unpack(o);
      if (!t[i]->is_contiguous() || t[i]->device() != dev) Py_RETURN_NONE;
    }
    auto is = [](const Tensor& x, ScalarType type, int64_t numel) {
      return x.scalar_type() == type && x.numel() == numel;
    };
    struct Linear {
      const int8_t* w;
      const float *bias, *sx, *sw, *so;
      int64_t n, k;
      size_t need;
    } l[kLinears];
    for (int i = 0; i < kLinears; ++i) {
      const Tensor* const* o = t + i * kEach;
      const int64_t k = i == 3 ? l[2].n : hidden, rows = o[0]->dim() == 2 ? o[0]->size(0) : 0;
      if (rows <= 0 || !is(*o[0], ScalarType::Char, rows * k) || (i == 0 ? rows != 3 * hidden : i != 2 && rows != hidden) ||
          !is(*o[1], ScalarType::Float, rows) || !is(*o[2], ScalarType::Float, 1) ||
          !is(*o[3], ScalarType::Float, rows) || !is(*o[4], ScalarType::Float, 1))
        Py_RETURN_NONE;
      l[i] = {(const int8_t*)in(*o[0]), (const float*)in(*o[1]), (const float*)in(*o[2]), (const float*)in(*o[3]),
              (const float*)in(*o[4]), rows, k, dq8_qgemm_workspace_bytes_zp(M, rows, k, 0, 1, 0, 0)};
    }
    const Tensor* const* last = t + kLinears * kEach;
    if (!is(*last[0], ScalarType::Char, 256) || !is(*last[5], ScalarType::Int, 1)) Py_RETURN_NONE;
    for (int i = 1; i < 5; ++i)
      if (!is(*last[i], ScalarType::Float, hidden)) Py_RETURN_NONE;
    const void* table = in(*last[0]);
    const float *g1 = (const float*)in(*last[1]), *b1 = (const float*)in(*last[2]);
    const float *g2 = (const float*)in(*last[3]), *b2 = (const float*)in(*last[4]);
    const int32_t* zero = (const int32_t*)in(*last[5]);
    const Tensor h = dense(h0);
    const float* x = (const float*)in(h);
    // the int8 input of each linear and the merged projection; the f32 results: the sum in front of
    // either layer norm (the second overwrites the first, which has been read by then), the first norm,
    // the layer
    Tensor q[kLinears + 1], y[3];
    for (int i = 0; i < kLinears; ++i) q[i] = empty({M, l[i].k}, ScalarType::Char, dev);
    q[kLinears] = empty({M, 3 * hidden}, ScalarType::Char, dev);
    for (int i = 0; i < 2; ++i) y[i] = empty({M, hidden}, ScalarType::Float, dev);
    y[2] = empty(h.sizes(), ScalarType::Float, dev);
    int8_t* qp[kLinears + 1];
    float* yp[3];
    for (int i = 0; i <= kLinears; ++i) qp[i] = (int8_t*)inout(q[i]);
    for (int i = 0; i < 3; ++i) yp[i] = (float*)inout(y[i]);
    size_t need = 0;
    for (const Linear& i : l) need = std::max(need, i.need);
    Tensor ws;
    if (need) ws = empty({(int64_t)need}, ScalarType::Byte, dev);
    void* wsp = inout(ws);
    void* st = stream();
    const char* what = "";
    int failed = 0;
    {
      const dq8::Unlocked unlocked;
      auto ok = [&](const char* name, int status) {
        what = name;
        failed = status;
        return status == 0;
      };
      auto linear = [&](int i, void* out, int epilogue, const dq8_postops_t* post) {
        return ok("dq8_qgemm", dq8_qgemm_fused(qp[i], l[i].k, l[i].w, l[i].k, out, l[i].n, M, l[i].n, l[i].k, 0, 1,
                                               epilogue, l[i].bias, DQ8_BIAS_F32, l[i].sx, 1, l[i].sw, l[i].n,
                                               l[i].so, 1, 0, 0, 0, wsp, l[i].need, post, st));
      };
      dq8_postops_t gelu = {}, add_x = {}, add_h1 = {};
      gelu.table = table;
      add_x.residual = x;
      add_x.residual_kind = DQ8_RESIDUAL_F32;
      add_x.ldr = hidden;
      add_h1 = add_x;
      add_h1.residual = yp[1];
      ok("dq8_quantize", dq8_quantize_ex(x, DQ8_DTYPE_F32, qp[0], DQ8_I8, 1, 1, M * hidden, l[0].sx, zero, 1, -128,
                                         127, DQ8_ROUND_HALF_TO_EVEN, st)) &&
          linear(0, qp[kLinears], DQ8_EPI_REQUANT_CPU, nullptr) &&
          ok("dq8_attention_i8",
             dq8_attention_i8(qp[kLinears], l[0].so, batch, seq, heads, 64, nullptr, qp[1], l[1].sx, st)) &&
          linear(1, yp[0], DQ8_EPI_REQUANT_CPU_DEQUANT_F32, &add_x) &&
          ok("dq8_layernorm_f32",
             dq8_layernorm_f32(yp[0], M, hidden, g1, b1, eps, yp[1], qp[2], l[2].sx, st)) &&
          linear(2, qp[3], DQ8_EPI_REQUANT_CPU, &gelu) &&
          linear(3, yp[0], DQ8_EPI_REQUANT_CPU_DEQUANT_F32, &add_h1) &&
          ok("dq8_layernorm_f32", dq8_layernorm_f32(yp[0], M, hidden, g2, b2, eps, yp[2], nullptr, nullptr, st));
    }
    check(failed, what);
    return THPVariable_Wrap(y[2]);
  });
}

PyMethodDef kMethods[] = {
#define DQ8_METHOD(name, fn) {name, (PyCFunction)(void (*)(void))fn, METH_FASTCALL, nullptr}
    DQ8_METHOD("quantize", py_quantize),
    DQ8_METHOD("dequantize", py_dequantize),
    DQ8_METHOD("fake_quant", py_fake_quant),
    DQ8_METHOD("minmax", py_minmax),
    DQ8_METHOD("observe", py_observe),
    DQ8_METHOD("lut8", py_lut8),
    DQ8_METHOD("weight_only_qgemm", py_weight_only),
    DQ8_METHOD("qgemm", py_qgemm),
    DQ8_METHOD("qlinear_f32", py_qlinear_f32),
    DQ8_METHOD("qconv2d", py_qconv2d),
    DQ8_METHOD("attention", py_attention),
    DQ8_METHOD("layer_norm", py_layer_norm),
    DQ8_METHOD("encoder_layer", py_encoder_layer),
#undef DQ8_METHOD
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_torch_calls", nullptr, -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_calls(void) { return PyModule_Create(&kModule); }
