// Calls into libakv_amd.so for the Python wrappers, without ctypes: the
// argument conversions follow from the declarations in akv_amd.h, and the
// functions' addresses come from the library that _lib loaded.
//
// ctypes took 3-4 us for the 30-odd arguments of an entry point (about a third
// of a wrapper's host time, and the small calls are bound by that time); these
// conversions take about 0.5 us.  Arguments that are not plain ints, floats or
// None go to the ctypes function, whose errors stand.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/akv_amd.h"

namespace {

template <typename T>
bool convert(PyObject* o, T* out) {
  if constexpr (std::is_pointer_v<T>) {
    if (o == Py_None) {
      *out = nullptr;
      return true;
    }
    if (!PyLong_Check(o)) return false;
    *out = reinterpret_cast<T>(static_cast<uintptr_t>(PyLong_AsUnsignedLongLongMask(o)));
    return true;
  } else if constexpr (std::is_floating_point_v<T>) {
    if (!PyFloat_Check(o)) return false;
    *out = static_cast<T>(PyFloat_AS_DOUBLE(o));
    return true;
  } else {
    if (!PyLong_Check(o)) return false;
    *out = static_cast<T>(PyLong_AsUnsignedLongLongMask(o));
    return true;
  }
}

template <typename... A, size_t... I>
bool convert_all(PyObject* const* args, std::tuple<A...>* to, std::index_sequence<I...>) {
  return (convert(args[I], &std::get<I>(*to)) && ...);
}

template <typename R, typename... A>
PyObject* invoke(R (*fn)(A...), PyObject* slow, PyObject* const* args, Py_ssize_t n) {
  if (!fn) {
    PyErr_SetString(PyExc_RuntimeError, "akv_amd native call before its library was loaded");
    return nullptr;
  }
  std::tuple<A...> v;
  if (n != static_cast<Py_ssize_t>(sizeof...(A)) || !convert_all(args, &v, std::index_sequence_for<A...>{}))
    return PyObject_Vectorcall(slow, args, n, nullptr);
  R r;
  Py_BEGIN_ALLOW_THREADS;
  r = std::apply(fn, v);
  Py_END_ALLOW_THREADS;
  return PyLong_FromLongLong(static_cast<long long>(r));
}

#define AKV_CALLS(X)                      \
  X(akv_reposition_kv_layers_gated)       \
  X(akv_compact_rows)                     \
  X(akv_compact_pages)                    \
  X(akv_bind_occurrences)                 \
  X(akv_decode_indices)                   \
  X(akv_window_lengths)                   \
  X(akv_build_indptr)                     \
  X(akv_write_row_slots)                  \
  X(akv_write_extend_rows)                \
  X(akv_decode_attention_workspace_bytes) \
  X(akv_decode_attention)                 \
  X(akv_context_attention)                \
  X(akv_context_attention_sized)          \
  X(akv_context_attention_split)          \
  X(akv_context_attention_split_bytes)    \
  X(akv_copy_kv_rows)                     \
  X(akv_gather_slots)

#define AKV_DEFINE(name)                                                   \
  decltype(&name) fn_##name = nullptr;                                     \
  PyObject* slow_##name = nullptr;                                         \
  PyObject* call_##name(PyObject*, PyObject* const* args, Py_ssize_t n) {  \
    return invoke(fn_##name, slow_##name, args, n);                        \
  }
AKV_CALLS(AKV_DEFINE)

// bind(name, address, ctypes function)
PyObject* bind(PyObject*, PyObject* args) {
  const char* name;
  unsigned long long address;
  PyObject* slow;
  if (!PyArg_ParseTuple(args, "sKO", &name, &address, &slow)) return nullptr;
#define AKV_BIND(x)                                                                   \
  if (std::strcmp(name, #x) == 0) {                                                   \
    fn_##x = reinterpret_cast<decltype(&x)>(static_cast<uintptr_t>(address));         \
    Py_INCREF(slow);                                                                  \
    Py_XSETREF(slow_##x, slow);                                                       \
    Py_RETURN_NONE;                                                                   \
  }
  AKV_CALLS(AKV_BIND)
  PyErr_Format(PyExc_ValueError, "no such call: %s", name);
  return nullptr;
}

PyObject* names(PyObject*, PyObject*) {
  PyObject* list = PyList_New(0);
  if (!list) return nullptr;
#define AKV_NAME(x)                                       \
  {                                                       \
    PyObject* s = PyUnicode_FromString(#x);               \
    if (!s || PyList_Append(list, s) < 0) {               \
      Py_XDECREF(s);                                      \
      Py_DECREF(list);                                    \
      return nullptr;                                     \
    }                                                     \
    Py_DECREF(s);                                         \
  }
  AKV_CALLS(AKV_NAME)
  return list;
}

#define AKV_METHOD(x) {#x, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(call_##x)), METH_FASTCALL, nullptr},
PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    {"names", names, METH_NOARGS, nullptr},
    AKV_CALLS(AKV_METHOD){nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }
