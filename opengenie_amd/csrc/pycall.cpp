// _native: the entry points of libopengenie_amd.so as functions of a CPython
// module. A call through ctypes converts each of its 7 to 25 arguments through
// a Python-level type object (~2 us a call beside the launch's own ~3 us); here
// the conversions are compiled from the declarations in opengenie_amd.h.
//
// Pointers are ints (addresses) or None, int64_t arrays (strides) a tuple of
// ints or any object with a buffer of int64_t (a ctypes array), numbers plain
// ints and floats. The GIL is released during the call, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/opengenie_amd.h"

namespace {

template <typename T, typename = void>
struct Arg;

template <typename T>
struct Arg<T, std::enable_if_t<std::is_integral_v<T>>> {
  T v{};
  bool get(PyObject* o) {
    const long long x = PyLong_AsLongLong(o);
    if (x == -1 && PyErr_Occurred()) return false;
    v = (T)x;
    if ((long long)v != x) {
      PyErr_SetString(PyExc_OverflowError, "integer argument out of range");
      return false;
    }
    return true;
  }
};

template <>
struct Arg<float> {
  float v = 0.0f;
  bool get(PyObject* o) {
    const double x = PyFloat_AsDouble(o);
    if (x == -1.0 && PyErr_Occurred()) return false;
    v = (float)x;
    return true;
  }
};

template <typename T>
struct Arg<T*, std::enable_if_t<!std::is_same_v<T, const int64_t>>> {
  T* v = nullptr;
  bool get(PyObject* o) {
    if (o == Py_None) return true;
    v = (T*)PyLong_AsVoidPtr(o);
    return !(v == nullptr && PyErr_Occurred());
  }
};

template <>
struct Arg<const int64_t*> {
  static constexpr Py_ssize_t kMax = 8;
  const int64_t* v = nullptr;
  int64_t buf[kMax] = {};  // (as long as any array argument is read; none is longer than 5)
  bool get(PyObject* o) {
    if (o == Py_None) return true;
    v = buf;
    if (PyTuple_Check(o)) {
      const Py_ssize_t n = PyTuple_GET_SIZE(o);
      if (n > kMax) return too_long();
      for (Py_ssize_t i = 0; i < n; ++i) {
        buf[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(o, i));
        if (buf[i] == -1 && PyErr_Occurred()) return false;
      }
      return true;
    }
    Py_buffer b;
    if (PyObject_GetBuffer(o, &b, PyBUF_SIMPLE) != 0) return false;
    const bool fits = b.len <= (Py_ssize_t)sizeof(buf);
    if (fits) __builtin_memcpy(buf, b.buf, (size_t)b.len);
    PyBuffer_Release(&b);
    return fits || too_long();
  }
  static bool too_long() {
    PyErr_SetString(PyExc_ValueError, "array argument too long");
    return false;
  }
};

template <auto F>
struct Call;

template <typename R, typename... A, R (*F)(A...)>
struct Call<F> {
  template <size_t... I>
  static PyObject* run(PyObject* const* args, std::index_sequence<I...>) {
    std::tuple<Arg<A>...> a;
    if (!(std::get<I>(a).get(args[I]) && ...)) return nullptr;
    R r;
    Py_BEGIN_ALLOW_THREADS
    r = F(std::get<I>(a).v...);
    Py_END_ALLOW_THREADS
    return PyLong_FromLongLong((long long)r);
  }
  static PyObject* fast(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != (Py_ssize_t)sizeof...(A)) {
      PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", (Py_ssize_t)sizeof...(A), n);
      return nullptr;
    }
    return run(args, std::index_sequence_for<A...>{});
  }
};

#define OGA_FN(name) \
  { #name, (PyCFunction)(void (*)(void))Call<name>::fast, METH_FASTCALL, nullptr }

PyMethodDef kMethods[] = {
    OGA_FN(oga_adazero_from_ada),
    OGA_FN(oga_adazero_from_ada_fp8),
    OGA_FN(oga_adazero),
    OGA_FN(oga_adaln_affine_from_ada),
    OGA_FN(oga_mul_from_ada),
    OGA_FN(oga_residual_gate_from_ada),
    OGA_FN(oga_residual_gate_bias_from_ada),
    OGA_FN(oga_residual_gate_adazero_from_ada),
    OGA_FN(oga_residual_gate_bf16),
    OGA_FN(oga_bias_add_bf16),
    OGA_FN(oga_head_gate_mul_bf16),
    OGA_FN(oga_fp8_quantize_e4m3),
    OGA_FN(oga_gelu_tanh_fp8_quantize_e4m3),
    OGA_FN(oga_fp8_per_head_workspace_bytes),
    OGA_FN(oga_fp8_quantize_per_head),
    OGA_FN(oga_video_qk_rmsnorm_rope),
    OGA_FN(oga_video_rmsnorm_rope),
    OGA_FN(oga_rmsnorm),
    OGA_FN(oga_video_qk_bias_rmsnorm_rope),
    OGA_FN(oga_video_qkv_rmsnorm_rope_pack),
    OGA_FN(oga_fp8_linear_workspace_bytes),
    OGA_FN(oga_fp8_linear_dt_ws),
    OGA_FN(oga_fp8_linear_grouped_ws),
    OGA_FN(oga_attention_workspace_bytes),
    OGA_FN(oga_attention_ws),
    OGA_FN(oga_attention_e4m3_out_ws),
    OGA_FN(oga_fp8_dequant_per_head),
    OGA_FN(oga_attention_fp8_workspace_bytes),
    OGA_FN(oga_attention_fp8_ws),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", "Entry points of libopengenie_amd.so.", -1, kMethods};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&kModule); }
