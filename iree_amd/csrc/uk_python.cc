// The C-ABI functions that a program calls once per matmul as builtins of CPython,
// in place of the ctypes functions of the same names (iree_amd/_lib.py): the same
// positional arguments and the same status, without ctypes' conversion object for
// every argument, which took 0.75 us of a call of mmt4d where this takes 0.15.
//
// Plain arguments (int, float, None for a null pointer) are converted here; a call
// with any other argument, or another number of them, goes to the ctypes function as
// it stands, so everything that was accepted is, and what is refused is refused by
// the same code. The interpreter lock is released around the function, as ctypes does.
// The module links against neither the library nor torch: bind() receives addresses.
// It keeps to the limited API, so that one binary serves every CPython from 3.10 on.
#define PY_SSIZE_T_CLEAN
#define Py_LIMITED_API 0x030A0000
#include <Python.h>

#include <stdint.h>
#include <string.h>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/iree_amd_uk.h"

namespace {

struct Bound {
  void* function;
  PyObject* ctypes_function;
};

// True when `v` was converted (ints wider than the parameter keep their low bits, as
// with ctypes).
template <typename T>
bool convert(PyObject* v, T& out) {
  if constexpr (std::is_pointer<T>::value) {
    if (v == Py_None) { out = nullptr; return true; }
    if (!PyLong_CheckExact(v)) return false;
    out = (T)(uintptr_t)PyLong_AsUnsignedLongLongMask(v);
  } else if constexpr (std::is_floating_point<T>::value) {
    if (!PyFloat_CheckExact(v)) return false;
    out = (T)PyFloat_AsDouble(v);
  } else {
    if (!PyLong_CheckExact(v)) return false;
    out = (T)PyLong_AsUnsignedLongLongMask(v);
  }
  return true;
}

PyObject* pass_on(const Bound* b, PyObject* const* args, Py_ssize_t n) {
  PyObject* tuple = PyTuple_New(n);
  if (!tuple) return nullptr;
  for (Py_ssize_t i = 0; i < n; ++i) {
    Py_INCREF(args[i]);
    PyTuple_SetItem(tuple, i, args[i]);      // (takes the reference)
  }
  PyObject* result = PyObject_CallObject(b->ctypes_function, tuple);
  Py_DECREF(tuple);
  return result;
}

template <typename Function>
struct Entry;
template <typename... A>
struct Entry<int (*)(A...)> {
  template <size_t... I>
  static PyObject* run(const Bound* b, PyObject* const* args, Py_ssize_t n, std::index_sequence<I...>) {
    std::tuple<std::remove_const_t<A>...> a;
    if (n != (Py_ssize_t)sizeof...(A) || !(convert(args[I], std::get<I>(a)) && ...)) return pass_on(b, args, n);
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = ((int (*)(A...))b->function)(std::get<I>(a)...);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(status);
  }
  static PyObject* call(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    const Bound* b = (const Bound*)PyCapsule_GetPointer(self, nullptr);
    return b ? run(b, args, n, std::index_sequence_for<A...>()) : nullptr;
  }
};

// (M0, N0, K0) of iree_amd_uk_query_matmul_tile_sizes, None where it has a status to
// report or the arguments are not plain: the caller then goes through ctypes.
PyObject* query(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  const Bound* b = (const Bound*)PyCapsule_GetPointer(self, nullptr);
  if (!b) return nullptr;
  uint32_t operation;
  iree_amd_uk_index_t M, N, K;
  if (n != 4 || !convert(args[0], operation) || !convert(args[1], M) || !convert(args[2], N) || !convert(args[3], K))
    Py_RETURN_NONE;
  iree_amd_uk_matmul_tile_t t;
  memset(&t, 0, sizeof t);
  if (((decltype(&iree_amd_uk_query_matmul_tile_sizes))b->function)(operation, M, N, K, &t) != 0) Py_RETURN_NONE;
  return Py_BuildValue("(iii)", (int)t.M, (int)t.N, (int)t.K);
}

#define UK_ENTRY(name) {#name, (PyCFunction)(void (*)(void))Entry<decltype(&name)>::call, METH_FASTCALL, nullptr}
PyMethodDef g_entries[] = {
    UK_ENTRY(iree_amd_uk_mmt4d),
    UK_ENTRY(iree_amd_uk_pack),
    UK_ENTRY(iree_amd_uk_unpack),
    UK_ENTRY(iree_amd_uk_mmt4d_unpack),
    UK_ENTRY(iree_amd_uk_matmul_packed_rhs),
    UK_ENTRY(iree_amd_uk_batch_mmt4d_unpack),
    UK_ENTRY(iree_amd_uk_batch_matmul_packed_rhs),
    UK_ENTRY(iree_amd_uk_matmul_data_tiled),
    UK_ENTRY(iree_amd_uk_dequant_matmul_i4),
    UK_ENTRY(iree_amd_uk_quantize_f16_to_f8e4m3),
    UK_ENTRY(iree_amd_uk_quantize_pack_f8e4m3),
    UK_ENTRY(iree_amd_uk_silu_mul_quantize_tiled),
    UK_ENTRY(iree_amd_uk_mmt4d_silu_mul_f8e4m3),
    UK_ENTRY(iree_amd_uk_scale_f32),
    {"iree_amd_uk_query_matmul_tile_sizes", (PyCFunction)(void (*)(void))query, METH_FASTCALL, nullptr},
};

// names(): the functions that there is a builtin for.
PyObject* names(PyObject*, PyObject*) {
  PyObject* list = PyList_New(0);
  for (const PyMethodDef& e : g_entries) {
    PyObject* name = list ? PyUnicode_FromString(e.ml_name) : nullptr;
    if (!name || PyList_Append(list, name)) {
      Py_XDECREF(name);
      Py_XDECREF(list);
      return nullptr;
    }
    Py_DECREF(name);
  }
  return list;
}

void release(PyObject* capsule) {
  Bound* b = (Bound*)PyCapsule_GetPointer(capsule, nullptr);
  if (!b) return;
  Py_XDECREF(b->ctypes_function);
  delete b;
}

// bind(name, address, ctypes function): the builtin.
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  const char* name = n == 3 ? PyUnicode_AsUTF8AndSize(args[0], nullptr) : nullptr;
  void* function = name && PyLong_CheckExact(args[1]) ? PyLong_AsVoidPtr(args[1]) : nullptr;
  if (!function) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "bind(name, address, function) expected");
    return nullptr;
  }
  for (PyMethodDef& e : g_entries) {
    if (strcmp(e.ml_name, name)) continue;
    Bound* b = new Bound{function, args[2]};
    Py_INCREF(args[2]);
    PyObject* capsule = PyCapsule_New(b, nullptr, release);
    if (!capsule) {
      Py_DECREF(args[2]);
      delete b;
      return nullptr;
    }
    PyObject* made = PyCFunction_New(&e, capsule);
    Py_DECREF(capsule);
    return made;
  }
  PyErr_Format(PyExc_KeyError, "no builtin of %s", name);
  return nullptr;
}

PyMethodDef g_methods[] = {
    {"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, nullptr},
    {"names", names, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "uk_python", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_uk_python(void) { return PyModule_Create(&g_module); }
