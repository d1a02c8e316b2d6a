// CPython module _bfa_entry: the C ABI's entry points as vector-call functions.
//
// Each entry takes the C function's arguments in order: int for int and int64_t,
// int or None for pointers, a number for float, and what ctypes takes in their place
// (its scalars, arrays, pointers and byref(), an object's _as_parameter_); it returns
// the C result.  An int that the C type does not hold raises OverflowError.  ctypes
// converts the 50 arguments of a fused call through Python-level argument types in
// about 5 us, as long as two kernel launches; these functions take 1.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <limits>
#include <tuple>
#include <type_traits>
#include <utility>

#include "braidinfer_amd.h"

namespace {

// Address that ctypes passes for an array, a pointer, byref() or bytes:
// ctypes.cast(o, ctypes.c_void_p).value, a new reference; null with a TypeError.
PyObject* ctypes_address(PyObject* o) {
  PyObject* address = nullptr;
  if (PyObject* ctypes = PyUnicode_Check(o) ? nullptr : PyImport_ImportModule("ctypes")) {
    PyObject* type = PyObject_GetAttrString(ctypes, "c_void_p");
    PyObject* pointer = type ? PyObject_CallMethod(ctypes, "cast", "OO", o, type) : nullptr;
    if (pointer) address = PyObject_GetAttrString(pointer, "value");
    Py_XDECREF(pointer);
    Py_XDECREF(type);
    Py_DECREF(ctypes);
  }
  if (!address) {
    PyErr_Clear();
    PyErr_Format(PyExc_TypeError, "an int, None or a ctypes object is required for a pointer, not %s",
                 Py_TYPE(o)->tp_name);
  }
  return address;
}

template <class T>
bool from_py(PyObject* o, T& v) {
  if (!PyLong_Check(o) && !PyFloat_Check(o) && o != Py_None) {
    // a ctypes scalar (c_void_p, c_float, ...) stands for its value
    for (const char* name : {"value", "_as_parameter_"}) {
      PyObject* value = PyObject_GetAttrString(o, name);
      if (!value) {
        PyErr_Clear();
        continue;
      }
      const bool plain = PyLong_Check(value) || PyFloat_Check(value) || value == Py_None;
      const bool ok = plain && from_py(value, v);
      Py_DECREF(value);
      if (plain) return ok;
    }
    if constexpr (std::is_pointer_v<T>) {
      PyObject* value = ctypes_address(o);
      const bool ok = value && from_py(value, v);
      Py_XDECREF(value);
      return ok;
    }
  }
  if constexpr (std::is_pointer_v<T>) {
    if (o == Py_None) {
      v = nullptr;
      return true;
    }
    v = static_cast<T>(PyLong_AsVoidPtr(o));
    return !(v == nullptr && PyErr_Occurred());
  } else if constexpr (std::is_floating_point_v<T>) {
    const double d = PyFloat_AsDouble(o);
    v = static_cast<T>(d);
    return !(d == -1.0 && PyErr_Occurred());
  } else {
    const long long x = PyLong_AsLongLong(o);
    if (x == -1 && PyErr_Occurred()) return false;
    if (x < std::numeric_limits<T>::min() || x > std::numeric_limits<T>::max()) {
      PyErr_Format(PyExc_OverflowError, "argument %lld does not fit a C %s", x, sizeof(T) == 4 ? "int" : "int64_t");
      return false;
    }
    v = static_cast<T>(x);
    return true;
  }
}

template <auto Fn>
struct Entry;

template <class R, class... A, R (*Fn)(A...)>
struct Entry<Fn> {
  static PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != static_cast<Py_ssize_t>(sizeof...(A))) {
      PyErr_Format(PyExc_TypeError, "this entry point takes %d arguments (%zd given)", static_cast<int>(sizeof...(A)), n);
      return nullptr;
    }
    return run(args, std::index_sequence_for<A...>{});
  }
  template <size_t... I>
  static PyObject* run(PyObject* const* args, std::index_sequence<I...>) {
    std::tuple<A...> t{};
    if (!(from_py(args[I], std::get<I>(t)) && ...)) return nullptr;
    R r;
    Py_BEGIN_ALLOW_THREADS
    r = Fn(std::get<I>(t)...);
    Py_END_ALLOW_THREADS
    return PyLong_FromLongLong(r);
  }
};

#define BFA_ENTRY(name) \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Entry<&name>::call)), METH_FASTCALL, nullptr}

PyMethodDef methods[] = {
    BFA_ENTRY(bfa_abi_version),
    BFA_ENTRY(bfa_set_tuning),
    BFA_ENTRY(bfa_get_tuning),
    BFA_ENTRY(bfa_rms_norm),
    BFA_ENTRY(bfa_add_rms_norm),
    BFA_ENTRY(bfa_rms_norm_f32),
    BFA_ENTRY(bfa_embedding),
    BFA_ENTRY(bfa_embedding_scaled),
    BFA_ENTRY(bfa_silu_and_mul),
    BFA_ENTRY(bfa_rotary_embedding),
    BFA_ENTRY(bfa_apply_rotary_emb),
    BFA_ENTRY(bfa_rerotate_paged_k),
    BFA_ENTRY(bfa_fused_rmsnorm_qkv_workspace_size),
    BFA_ENTRY(bfa_fused_rmsnorm_qkv),
    BFA_ENTRY(bfa_fused_rmsnorm_qkv_noalloc),
    BFA_ENTRY(bfa_fold_rmsnorm_weight),
    BFA_ENTRY(bfa_rmsnorm_row_scale),
    BFA_ENTRY(bfa_fused_rmsnorm_qkv_folded),
    BFA_ENTRY(bfa_rmsnorm_qkv_operand),
    BFA_ENTRY(bfa_qkv_projection),
    BFA_ENTRY(bfa_append_paged_kv),
    BFA_ENTRY(bfa_fused_rmsnorm_qkv_append_workspace_size),
    BFA_ENTRY(bfa_fused_rmsnorm_qkv_append),
    BFA_ENTRY(bfa_online_softmax_update),
    BFA_ENTRY(bfa_cascade_attention_workspace_size),
    BFA_ENTRY(bfa_cascade_attention),
    BFA_ENTRY(bfa_linear_workspace_size),
    BFA_ENTRY(bfa_linear),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_bfa_entry", "Entry points of libbraidinfer_amd.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__bfa_entry(void) { return PyModule_Create(&module); }
