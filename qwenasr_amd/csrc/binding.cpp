// Python binding of the C ABI (include/qasr.h) for torch tensors.
//
// What a call from Python cost was not the launch but the way to it: per
// argument a ctypes object, per tensor five Python-level checks, and the stream
// looked up through torch's Python classes; 10 us for a launch that takes
// 3.6 us of host time by itself (an empty kernel from a C++ loop). Here one
// extension call checks the tensors, reads their pointers and the current
// stream, and calls the entry point: 3.4 us per call (three small calls 29.6 ->
// 10.1 us of host time, a whole 0.6B decode step of 171 launches 1825 -> 709 us).
//
// The argument list of an entry point follows from its C prototype:
//   float* / int8_t* / int32_t* / uint16_t*  a tensor and the element count it
//                    must hold; None is a null pointer where the name ends in
//                    '?', and otherwise refused;
//   void* (not last) a tensor of any type, or None;
//   size_t, float    a number;
//   the last void*   the current stream (not passed).
// A tensor that fails a check is handed to the Python-side check, which raises
// the error with the argument's name. Nothing is remembered between calls.
#include <torch/csrc/autograd/python_variable.h>

#include <c10/hip/HIPStream.h>
#include <c10/util/SmallVector.h>

#include <cstdint>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/qasr.h"

namespace {

PyObject* g_need = nullptr;   // need(tensor, dtype, n, name): raises what is wrong
PyObject* g_raise = nullptr;  // raise_status(entry point, status): raises QasrError
PyObject* g_dtypes[4] = {};   // torch.float32, int8, int32, int16

struct PyError {};  // a Python exception is set

template <class T>
struct Elem;
template <>
struct Elem<float> {
  static constexpr int dtype = 0;
  static constexpr auto type = at::kFloat;
};
template <>
struct Elem<int8_t> {
  static constexpr int dtype = 1;
  static constexpr auto type = at::kChar;
};
template <>
struct Elem<int32_t> {
  static constexpr int dtype = 2;
  static constexpr auto type = at::kInt;
};
template <>
struct Elem<uint16_t> {
  static constexpr int dtype = 3;
  static constexpr auto type = at::kShort;
};

long long count_of(PyObject* o) {
  int overflow = 0;
  const long long n = PyLong_AsLongLongAndOverflow(o, &overflow);
  if (overflow) return overflow > 0 ? INT64_MAX : -1;
  if (n == -1 && PyErr_Occurred()) throw PyError();
  return n;
}

// The address that t.data_ptr() gives in Python (tensors the C++ side cannot
// look into: subclasses that dispatch in Python).
void* data_ptr_from_python(PyObject* o) {
  PyObject* p = PyObject_CallMethod(o, "data_ptr", nullptr);
  if (!p) throw PyError();
  void* v = PyLong_AsVoidPtr(p);
  Py_DECREF(p);
  if (!v && PyErr_Occurred()) throw PyError();
  return v;
}

template <class T>
T* tensor_arg(PyObject* o, PyObject* need, const char* name) {
  if (THPVariable_CheckExact(o) || THPVariable_Check(o)) {
    const at::Tensor& t = THPVariable_Unpack(o);
    if (t.is_cuda() && t.scalar_type() == Elem<T>::type && t.is_contiguous() && t.numel() >= count_of(need))
      return static_cast<T*>(t.data_ptr());
  }
  PyObject* r = PyObject_CallFunction(g_need, "OOOs", o, g_dtypes[Elem<T>::dtype], need, name);
  if (!r) throw PyError();
  Py_DECREF(r);
  return static_cast<T*>(data_ptr_from_python(o));
}

size_t size_arg(PyObject* o) {
  if (!PyLong_Check(o)) {
    PyErr_Format(PyExc_TypeError, "int expected instead of %s instance", Py_TYPE(o)->tp_name);
    throw PyError();
  }
  const unsigned long long v = PyLong_AsUnsignedLongLongMask(o);
  if (v == (unsigned long long)-1 && PyErr_Occurred()) throw PyError();
  return (size_t)v;
}

float float_arg(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw PyError();
  return (float)v;
}

struct Args {
  PyObject* const* at;
  Py_ssize_t left;
  const char* const* names;  // one per tensor argument, in order
  const char* fn;
  PyObject* next() {
    if (left == 0) {
      PyErr_Format(PyExc_TypeError, "%s: too few arguments", fn);
      throw PyError();
    }
    --left;
    return *at++;
  }
};

// One C argument from the Python arguments.
template <class T, bool Last>
T take(Args& a) {
  if constexpr (std::is_same_v<T, void*> && Last) {
    return static_cast<void*>(c10::hip::getCurrentHIPStream().stream());
  } else if constexpr (std::is_same_v<T, void*>) {
    PyObject* o = a.next();
    if (o == Py_None) return nullptr;
    if (THPVariable_Check(o)) return THPVariable_Unpack(o).data_ptr();
    PyErr_Format(PyExc_TypeError, "%s: expected a tensor or None", a.fn);
    throw PyError();
  } else if constexpr (std::is_pointer_v<T>) {
    using E = std::remove_const_t<std::remove_pointer_t<T>>;
    PyObject* o = a.next();
    PyObject* need = a.next();
    const char* name = *a.names++;
    if (o == Py_None && name[0] == '?') return nullptr;
    return tensor_arg<E>(o, need, name[0] == '?' ? name + 1 : name);
  } else if constexpr (std::is_same_v<T, float>) {
    return float_arg(a.next());
  } else {
    static_assert(std::is_same_v<T, size_t>);
    return size_arg(a.next());
  }
}

PyObject* finish(const char* fn, int rc) {
  if (rc == QASR_OK) Py_RETURN_NONE;
  PyObject* r = PyObject_CallFunction(g_raise, "si", fn, rc);
  Py_XDECREF(r);
  return nullptr;
}

// No C++ exception leaves an entry of this module.
template <class F>
PyObject* guarded(F&& f) {
  try {
    return f();
  } catch (const PyError&) {
  } catch (const std::exception& e) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what());
  } catch (...) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "unknown C++ exception");
  }
  return nullptr;
}

// The library is the one that ctypes loaded, so its addresses come from there.
template <class Tag>
struct Entry {
  static inline void* address = nullptr;
};

template <class Tag, class... A, size_t... I>
PyObject* call_entry(int (*)(A...), const char* fn, const char* const* names, PyObject* const* args, Py_ssize_t n,
                     std::index_sequence<I...>) {
  return guarded([&]() -> PyObject* {
    Args a{args, n, names, fn};
    std::tuple<A...> c{take<A, I + 1 == sizeof...(A)>(a)...};  // braces: left to right
    if (a.left != 0) {
      PyErr_Format(PyExc_TypeError, "%s: too many arguments", fn);
      throw PyError();
    }
    int rc;
    {
      PyThreadState* ts = PyEval_SaveThread();
      rc = std::apply(reinterpret_cast<int (*)(A...)>(Entry<Tag>::address), c);
      PyEval_RestoreThread(ts);
    }
    return finish(fn, rc);
  });
}

template <class R, class... A>
constexpr size_t arity(R (*)(A...)) {
  return sizeof...(A);
}

#define QASR_BIND(FN, ...)                                                                    \
  struct Tag_##FN {};                                                                         \
  PyObject* py_##FN(PyObject*, PyObject* const* args, Py_ssize_t n) {                         \
    static const char* const names[] = {__VA_ARGS__};                                         \
    using Fn = decltype(&::FN);                                                               \
    return call_entry<Tag_##FN>(Fn(nullptr), #FN, names, args, n,                             \
                                std::make_index_sequence<arity(Fn(nullptr))>());              \
  }

QASR_BIND(qasr_add_inplace_f32, "a", "b")
QASR_BIND(qasr_rms_norm_f32, "out", "x", "weight")
QASR_BIND(qasr_add_rms_norm_f32, "x", "delta", "weight", "out")
QASR_BIND(qasr_add_rms_norm_quant_f32, "x", "?delta", "weight", "?out", "q", "q_scales")
QASR_BIND(qasr_layer_norm_f32, "out", "x", "weight", "bias")
QASR_BIND(qasr_add_layer_norm_f32, "x", "delta", "weight", "bias", "out")
QASR_BIND(qasr_rms_norm_per_head_f32, "x", "weight")
QASR_BIND(qasr_apply_rope_neox_f32, "x", "cos_vals", "sin_vals")
QASR_BIND(qasr_head_rms_norm_rope_f32, "?q", "?k", "?q_norm_w", "?k_norm_w", "cos_tab", "sin_tab", "?positions")
QASR_BIND(qasr_head_rms_norm_rope_kv_f32, "?q", "?k", "?v", "?q_norm_w", "?k_norm_w", "cos", "sin", "?positions",
          "?k_cache", "?v_cache")
QASR_BIND(qasr_swiglu_multiply_f32, "out", "gate_up")
QASR_BIND(qasr_swiglu_split_f32, "out", "gate", "up")
QASR_BIND(qasr_silu_f32, "x")
QASR_BIND(qasr_gelu_tanh_f32, "x")
QASR_BIND(qasr_gelu_erf_f32, "x")
QASR_BIND(qasr_pe_add_f32, "x", "pe")
QASR_BIND(qasr_pe_add_layer_norm_f32, "x", "pe", "out", "weight", "bias")
QASR_BIND(qasr_embed_gather_f32, "out", "table", "ids")
QASR_BIND(qasr_embed_gather_bf16, "out", "table", "ids")
QASR_BIND(qasr_embed_gather_i8, "out", "w.data", "w.scales", "ids")
QASR_BIND(qasr_quantize_rows_i8, "q", "scales", "x")
QASR_BIND(qasr_linear_nobias_int8_f32, "y", "x", "w_int8", "scales")
QASR_BIND(qasr_linear_int8_f32, "y", "x", "w_int8", "scales", "?bias")
QASR_BIND(qasr_gate_up_swiglu_int8_f32, "out", "x", "w", "scales")
QASR_BIND(qasr_gate_up_swiglu_multiply_int8_f32, "out", "x", "w", "scales")
QASR_BIND(qasr_qkv_heads_int8_f32, "q", "k_cache", "v_cache", "wq", "wq.scales", "wk", "wk.scales", "wv", "wv.scales",
          "x", "q_norm_w", "k_norm_w", "cos", "sin")
QASR_BIND(qasr_rms_norm_qkv_heads_int8_f32, "q", "k_cache", "v_cache", "wq", "wq.scales", "wk", "wk.scales", "wv",
          "wv.scales", "hg", "ss", "x_norm", "q_norm_w", "k_norm_w", "cos", "sin")
QASR_BIND(qasr_linear_int8_residual_f32, "h", "ss", "?hg", "?gain", "x", "w", "scales")
QASR_BIND(qasr_rms_norm_gate_up_swiglu_multiply_int8_f32, "out", "hg", "ss", "x_norm", "w", "scales")
QASR_BIND(qasr_add_rms_norm_gate_up_swiglu_int8_f32, "out", "?h_out", "x", "?delta", "norm_w", "w", "scales")
QASR_BIND(qasr_gate_up_swiglu_w8a8, "out", "w.data", "w.scales", "xq", "x_scales")
QASR_BIND(qasr_gate_up_swiglu_w8a8_f32in, "out", "w.data", "w.scales", "x")
QASR_BIND(qasr_gate_up_swiglu_w8a8_packed, "out", "w.data", "w.scales", "xq", "x_scales")
QASR_BIND(qasr_linear_w8a8_packed, "y", "w.data", "w.scales", "xq", "x_scales")
QASR_BIND(qasr_qkv_heads_w8a8_packed, "q_out", "k_cache", "v_cache", "w.data", "w.scales", "xq", "x_scales",
          "q_norm_w", "k_norm_w", "cos", "sin", "positions")
QASR_BIND(qasr_digit_rows_f32, "digits", "exps", "x")
QASR_BIND(qasr_digit_rows_wide_f32, "digits", "exps", "x")
QASR_BIND(qasr_add_rms_norm_digits_f32, "x", "?delta", "weight", "?x_norm", "digits", "exps")
QASR_BIND(qasr_add_rms_norm_digits_wide_f32, "x", "?delta", "weight", "x_norm", "digits", "exps")
QASR_BIND(qasr_gate_up_swiglu_digits_wide_int8_f32, "out", "w.data", "w.scales", "digits", "exps", "?x")
QASR_BIND(qasr_qkv_heads_digits_wide_int8_f32, "q", "k_cache", "v_cache", "wq", "wq.scales", "wk", "wk.scales", "wv",
          "wv.scales", "digits", "exps", "?x", "q_norm_w", "k_norm_w", "cos", "sin")
QASR_BIND(qasr_causal_attention_f32, "out", "q", "?k", "?v")
QASR_BIND(qasr_causal_attention_split_f32, "out", "q", "?k", "?v", "workspace")
QASR_BIND(qasr_decode_attention_f32, "out", "q", "k", "v", "q_norm_w", "k_norm_w", "cos", "sin", "k_cache", "v_cache",
          "workspace")
QASR_BIND(qasr_decode_attention_linear_int8_f32, "y", "out", "q", "k", "v", "q_norm_w", "k_norm_w", "cos", "sin",
          "k_cache", "v_cache", "workspace", "w", "scales")
QASR_BIND(qasr_batched_decode_attention_f32, "out", "q", "k_cache", "v_cache", "positions", "?workspace", "?out_q",
          "?out_scales", "?order")
QASR_BIND(qasr_batched_decode_order_i32, "order", "positions")
QASR_BIND(qasr_argmax_rows_f32, "idx", "x")
QASR_BIND(qasr_lm_head_int8_argmax_f32, "idx", "logits", "x", "w", "scales")

// The launches of several matrices take lists: ys of tensors and ws of objects
// with data, scales and out_dim; ys[m] must hold rows * ws[m].out_dim elements.
struct Mats {
  Py_ssize_t n = 0;
  c10::SmallVector<float*, 4> y;
  c10::SmallVector<const int8_t*, 4> w;
  c10::SmallVector<const float*, 4> s;
  c10::SmallVector<size_t, 4> out;
};

struct Ref {  // an owned reference
  PyObject* o;
  explicit Ref(PyObject* p) : o(p) {
    if (!p) throw PyError();
  }
  ~Ref() { Py_DECREF(o); }
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
};

Mats take_mats(Args& a, PyObject* rows, PyObject* in_dim) {
  static PyObject* const kData = PyUnicode_InternFromString("data");
  static PyObject* const kScales = PyUnicode_InternFromString("scales");
  static PyObject* const kOut = PyUnicode_InternFromString("out_dim");
  Ref ys(PySequence_Fast(a.next(), "ys must be a sequence")), ws(PySequence_Fast(a.next(), "ws must be a sequence"));
  Mats m;
  m.n = PySequence_Fast_GET_SIZE(ys.o);
  if (m.n != PySequence_Fast_GET_SIZE(ws.o)) {
    PyErr_SetString(PyExc_ValueError, "one output per weight");
    throw PyError();
  }
  for (Py_ssize_t i = 0; i < m.n; ++i) {
    PyObject* w = PySequence_Fast_GET_ITEM(ws.o, i);
    Ref out(PyObject_GetAttr(w, kOut)), data(PyObject_GetAttr(w, kData)), scales(PyObject_GetAttr(w, kScales));
    Ref ny(PyNumber_Multiply(rows, out.o)), nw(PyNumber_Multiply(out.o, in_dim));
    m.y.push_back(tensor_arg<float>(PySequence_Fast_GET_ITEM(ys.o, i), ny.o, "y"));
    m.w.push_back(tensor_arg<int8_t>(data.o, nw.o, "w"));
    m.s.push_back(tensor_arg<float>(scales.o, out.o, "scales"));
    m.out.push_back(size_arg(out.o));
  }
  return m;
}

struct Tag_multi {};
struct Tag_norm_multi {};
struct Tag_digits {};

// (ys, ws, x, n_x, seq_len, in_dim)
PyObject* py_multi(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    static const char* const names[] = {"x"};
    const char* fn = "qasr_linear_nobias_int8_multi_f32";
    Args a{args, n, names, fn};
    if (n != 6) {
      PyErr_Format(PyExc_TypeError, "%s: takes 6 arguments", fn);
      throw PyError();
    }
    const Mats m = take_mats(a, args[4], args[5]);
    const float* x = take<const float*, false>(a);
    const size_t seq = size_arg(a.next()), in_dim = size_arg(a.next());
    void* st = take<void*, true>(a);
    int rc;
    {
      PyThreadState* ts = PyEval_SaveThread();
      rc = reinterpret_cast<decltype(&qasr_linear_nobias_int8_multi_f32)>(Entry<Tag_multi>::address)(
          (size_t)m.n, m.y.data(), m.w.data(), m.s.data(), m.out.data(), x, seq, in_dim, st);
      PyEval_RestoreThread(ts);
    }
    return finish(fn, rc);
  });
}

// (ys, ws, h_out, n, x, n, delta, n, norm_w, n, in_dim, eps)
PyObject* py_norm_multi(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    static const char* const names[] = {"?h_out", "x", "?delta", "norm_w"};
    const char* fn = "qasr_add_rms_norm_linear_nobias_int8_multi_f32";
    Args a{args, n, names, fn};
    if (n != 12) {
      PyErr_Format(PyExc_TypeError, "%s: takes 12 arguments", fn);
      throw PyError();
    }
    Ref one(PyLong_FromLong(1));
    const Mats m = take_mats(a, one.o, args[10]);
    float* h_out = take<float*, false>(a);
    const float* x = take<const float*, false>(a);
    const float* delta = take<const float*, false>(a);
    const float* norm_w = take<const float*, false>(a);
    const size_t in_dim = size_arg(a.next());
    const float eps = float_arg(a.next());
    void* st = take<void*, true>(a);
    int rc;
    {
      PyThreadState* ts = PyEval_SaveThread();
      rc = reinterpret_cast<decltype(&qasr_add_rms_norm_linear_nobias_int8_multi_f32)>(Entry<Tag_norm_multi>::address)(
          (size_t)m.n, m.y.data(), m.w.data(), m.s.data(), m.out.data(), h_out, x, delta, norm_w, in_dim, eps, st);
      PyEval_RestoreThread(ts);
    }
    return finish(fn, rc);
  });
}

// (ys, ws, digits, n, exps, n, x, n, seq_len, in_dim, residual, parts, rows); ys hold rows = parts * seq_len rows
PyObject* py_digits(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    static const char* const names[] = {"digits", "exps", "?x"};
    const char* fn = "qasr_linear_digits_wide_int8_f32";
    Args a{args, n, names, fn};
    if (n != 13) {
      PyErr_Format(PyExc_TypeError, "%s: takes 13 arguments", fn);
      throw PyError();
    }
    const Mats m = take_mats(a, args[12], args[9]);
    const int8_t* digits = take<const int8_t*, false>(a);
    const int32_t* exps = take<const int32_t*, false>(a);
    const float* x = take<const float*, false>(a);
    const size_t seq = size_arg(a.next()), in_dim = size_arg(a.next()), residual = size_arg(a.next());
    const size_t parts = size_arg(a.next());
    void* st = take<void*, true>(a);
    int rc;
    {
      PyThreadState* ts = PyEval_SaveThread();
      rc = reinterpret_cast<decltype(&qasr_linear_digits_wide_int8_f32)>(Entry<Tag_digits>::address)(
          (size_t)m.n, m.y.data(), m.w.data(), m.s.data(), m.out.data(), digits, exps, x, seq, in_dim, residual,
          parts, st);
      PyEval_RestoreThread(ts);
    }
    return finish(fn, rc);
  });
}

struct Bound {
  const char* name;
  PyCFunction fn;
  void** address;
};

#define QASR_ENTRY(FN) \
  { #FN, (PyCFunction)(void (*)(void))py_##FN, &Entry<Tag_##FN>::address }

Bound g_bound[] = {
    QASR_ENTRY(qasr_add_inplace_f32),
    QASR_ENTRY(qasr_rms_norm_f32),
    QASR_ENTRY(qasr_add_rms_norm_f32),
    QASR_ENTRY(qasr_add_rms_norm_quant_f32),
    QASR_ENTRY(qasr_layer_norm_f32),
    QASR_ENTRY(qasr_add_layer_norm_f32),
    QASR_ENTRY(qasr_rms_norm_per_head_f32),
    QASR_ENTRY(qasr_apply_rope_neox_f32),
    QASR_ENTRY(qasr_head_rms_norm_rope_f32),
    QASR_ENTRY(qasr_head_rms_norm_rope_kv_f32),
    QASR_ENTRY(qasr_swiglu_multiply_f32),
    QASR_ENTRY(qasr_swiglu_split_f32),
    QASR_ENTRY(qasr_silu_f32),
    QASR_ENTRY(qasr_gelu_tanh_f32),
    QASR_ENTRY(qasr_gelu_erf_f32),
    QASR_ENTRY(qasr_pe_add_f32),
    QASR_ENTRY(qasr_pe_add_layer_norm_f32),
    QASR_ENTRY(qasr_embed_gather_f32),
    QASR_ENTRY(qasr_embed_gather_bf16),
    QASR_ENTRY(qasr_embed_gather_i8),
    QASR_ENTRY(qasr_quantize_rows_i8),
    QASR_ENTRY(qasr_linear_nobias_int8_f32),
    QASR_ENTRY(qasr_linear_int8_f32),
    QASR_ENTRY(qasr_gate_up_swiglu_int8_f32),
    QASR_ENTRY(qasr_gate_up_swiglu_multiply_int8_f32),
    QASR_ENTRY(qasr_qkv_heads_int8_f32),
    QASR_ENTRY(qasr_rms_norm_qkv_heads_int8_f32),
    QASR_ENTRY(qasr_linear_int8_residual_f32),
    QASR_ENTRY(qasr_rms_norm_gate_up_swiglu_multiply_int8_f32),
    QASR_ENTRY(qasr_add_rms_norm_gate_up_swiglu_int8_f32),
    QASR_ENTRY(qasr_gate_up_swiglu_w8a8),
    QASR_ENTRY(qasr_gate_up_swiglu_w8a8_f32in),
    QASR_ENTRY(qasr_gate_up_swiglu_w8a8_packed),
    QASR_ENTRY(qasr_linear_w8a8_packed),
    QASR_ENTRY(qasr_qkv_heads_w8a8_packed),
    QASR_ENTRY(qasr_digit_rows_f32),
    QASR_ENTRY(qasr_digit_rows_wide_f32),
    QASR_ENTRY(qasr_add_rms_norm_digits_f32),
    QASR_ENTRY(qasr_add_rms_norm_digits_wide_f32),
    QASR_ENTRY(qasr_gate_up_swiglu_digits_wide_int8_f32),
    QASR_ENTRY(qasr_qkv_heads_digits_wide_int8_f32),
    QASR_ENTRY(qasr_causal_attention_f32),
    QASR_ENTRY(qasr_causal_attention_split_f32),
    QASR_ENTRY(qasr_decode_attention_f32),
    QASR_ENTRY(qasr_decode_attention_linear_int8_f32),
    QASR_ENTRY(qasr_batched_decode_attention_f32),
    QASR_ENTRY(qasr_batched_decode_order_i32),
    QASR_ENTRY(qasr_argmax_rows_f32),
    QASR_ENTRY(qasr_lm_head_int8_argmax_f32),
    {"qasr_linear_nobias_int8_multi_f32", (PyCFunction)(void (*)(void))py_multi, &Entry<Tag_multi>::address},
    {"qasr_add_rms_norm_linear_nobias_int8_multi_f32", (PyCFunction)(void (*)(void))py_norm_multi,
     &Entry<Tag_norm_multi>::address},
    {"qasr_linear_digits_wide_int8_f32", (PyCFunction)(void (*)(void))py_digits, &Entry<Tag_digits>::address},
};
constexpr size_t kBound = sizeof(g_bound) / sizeof(g_bound[0]);
PyMethodDef g_defs[kBound];

// setup(address_of, need, raise_status, dtypes) -> {name: function}. address_of
// gives the loaded library's address of an entry point.
PyObject* py_setup(PyObject*, PyObject* args) {
  PyObject *address_of, *need, *raise_status, *dtypes;
  if (!PyArg_ParseTuple(args, "OOOO!", &address_of, &need, &raise_status, &PyTuple_Type, &dtypes)) return nullptr;
  if (PyTuple_GET_SIZE(dtypes) != 4) {
    PyErr_SetString(PyExc_ValueError, "four dtypes");
    return nullptr;
  }
  PyObject* out = PyDict_New();
  if (!out) return nullptr;
  for (size_t i = 0; i < kBound; ++i) {
    PyObject* p = PyObject_CallFunction(address_of, "s", g_bound[i].name);
    if (!p) {
      Py_DECREF(out);
      return nullptr;
    }
    *g_bound[i].address = PyLong_AsVoidPtr(p);
    Py_DECREF(p);
    if (!*g_bound[i].address) {
      if (!PyErr_Occurred()) PyErr_Format(PyExc_ImportError, "no entry point %s", g_bound[i].name);
      Py_DECREF(out);
      return nullptr;
    }
    g_defs[i] = PyMethodDef{g_bound[i].name, g_bound[i].fn, METH_FASTCALL, nullptr};
    PyObject* f = PyCFunction_New(&g_defs[i], nullptr);
    if (!f || PyDict_SetItemString(out, g_bound[i].name, f) != 0) {
      Py_XDECREF(f);
      Py_DECREF(out);
      return nullptr;
    }
    Py_DECREF(f);
  }
  Py_INCREF(need);
  Py_XSETREF(g_need, need);
  Py_INCREF(raise_status);
  Py_XSETREF(g_raise, raise_status);
  for (int i = 0; i < 4; ++i) {
    PyObject* d = PyTuple_GET_ITEM(dtypes, i);
    Py_INCREF(d);
    Py_XSETREF(g_dtypes[i], d);
  }
  return out;
}

PyMethodDef g_methods[] = {{"setup", py_setup, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding() { return PyModule_Create(&g_module); }
