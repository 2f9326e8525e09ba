// The compute entry points of the C ABI as Python functions of integers and floats, for the calls
// that litert_amd.fully_connected makes per op. A decode call's kernel takes 3 to 10 us, and
// through ctypes the host's part of it was longer: every pointer an object of its own, every
// argument converted by a callback. Here an argument is one PyLong read, its type taken from
// the header's declaration. A pointer is an integer address or None.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <limits>
#include <tuple>
#include <type_traits>
#include <utility>

#include "litert_amd_fc.h"

namespace {

template <typename T>
bool Convert(PyObject* o, T* out) {
  if constexpr (std::is_pointer_v<T>) {
    if (o == Py_None) {
      *out = nullptr;
      return true;
    }
    *out = static_cast<T>(PyLong_AsVoidPtr(o));
  } else if constexpr (std::is_floating_point_v<T>) {
    *out = static_cast<T>(PyFloat_AsDouble(o));
  } else if constexpr (std::is_unsigned_v<T>) {
    *out = static_cast<T>(PyLong_AsSize_t(o));
  } else {
    const long long v = PyLong_AsLongLong(o);
    if (!PyErr_Occurred() && (v < std::numeric_limits<T>::min() || v > std::numeric_limits<T>::max())) {
      PyErr_SetString(PyExc_OverflowError, "argument does not fit its C type");
    }
    *out = static_cast<T>(v);
  }
  return PyErr_Occurred() == nullptr;
}

template <typename R, typename... A, size_t... I>
PyObject* CallWith(R (*fn)(A...), PyObject* const* args, std::index_sequence<I...>) {
  std::tuple<A...> values;
  if (!(Convert(args[I], &std::get<I>(values)) && ...)) return nullptr;
  R result;
  Py_BEGIN_ALLOW_THREADS
  result = fn(std::get<I>(values)...);
  Py_END_ALLOW_THREADS
  if constexpr (std::is_unsigned_v<R>) {
    return PyLong_FromSize_t(result);
  } else {
    return PyLong_FromLongLong(result);
  }
}

template <typename R, typename... A>
PyObject* Call(R (*fn)(A...), PyObject* const* args, Py_ssize_t count) {
  if (count != static_cast<Py_ssize_t>(sizeof...(A))) {
    return PyErr_Format(PyExc_TypeError, "expected %zu arguments, got %zd", sizeof...(A), count);
  }
  return CallWith(fn, args, std::index_sequence_for<A...>{});
}

template <auto FN>
PyObject* Method(PyObject*, PyObject* const* args, Py_ssize_t count) {
  return Call(FN, args, count);
}

#define LRTFC_METHOD(name) \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Method<&name>)), METH_FASTCALL, nullptr}

PyMethodDef kMethods[] = {
    LRTFC_METHOD(lrtfc_fc_int8_packed),
    LRTFC_METHOD(lrtfc_fc_int8),
    LRTFC_METHOD(lrtfc_fc_hybrid_fused_max_batches),
    LRTFC_METHOD(lrtfc_fc_hybrid_packed),
    LRTFC_METHOD(lrtfc_fc_hybrid_packed_workspace),
    LRTFC_METHOD(lrtfc_fc_hybrid),
    LRTFC_METHOD(lrtfc_activation_workspace_bytes),
    LRTFC_METHOD(lrtfc_fc_blockwise_int4_preferred_form),
    LRTFC_METHOD(lrtfc_fc_blockwise_int4_packed),
    LRTFC_METHOD(lrtfc_batch_quantize_floats),
    LRTFC_METHOD(lrtfc_fc_blockwise_int4_packed_quantized),
    LRTFC_METHOD(lrtfc_fc_blockwise_int4_gemm_workspace_bytes),
    LRTFC_METHOD(lrtfc_fc_blockwise_int4_gemm),
    LRTFC_METHOD(lrtfc_fc_blockwise_int4_gemm_nibbles),
    LRTFC_METHOD(lrtfc_fc_hybrid_int4_per_channel_nibbles_max_batches),
    LRTFC_METHOD(lrtfc_fc_hybrid_int4_per_channel_nibbles),
    LRTFC_METHOD(lrtfc_fc_hybrid_int4_per_channel_packed),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "litert_amd_calls", nullptr, -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_litert_amd_calls() { return PyModule_Create(&kModule); }
