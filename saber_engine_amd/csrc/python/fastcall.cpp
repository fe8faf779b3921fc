// The operator entry points of include/saber_iu8.h as vectorcall functions for the Python binding (iu8.py).
//
// An operator is a launch, 5 us on the card for a decode linear, and is called from a serving loop: a call that takes longer
// on the host than its kernel is what the loop waits for. ctypes converts a dozen arguments one Python object at a time, 1.7 us
// a call; here an argument is read by the type the header declares, 0.7 us with the descriptor's layout. (With the layout's
// share, util.h: a one-row linear of 5120 x 5120 in a loop of calls 7.5-8.1 -> 6.5-7.2 us, its kernel 5; 16 rows, quantiser and
// GEMM, 11.6-12.7 -> 9.7-11.0.) The conversions are ctypes' own for what a caller
// passes: a pointer is an int or None, a number an int, a float a float, each taken modulo its width; the routed operators'
// tables are the structure itself (an address in their place is refused, as ctypes refuses it). Anything else in an argument's
// place (a ctypes object, a bool, another count of arguments) sends the whole call, its arguments as they came, to the ctypes
// function of the same name, which converts or refuses them. The interpreter lock is released around the call, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "../../../include/saber_iu8.h"

namespace {

PyObject *tables_type = nullptr;  // the binding's saber_iu8_moe_tables

template <class T>
bool take(PyObject *o, T &v) {
  if constexpr (std::is_same_v<T, const saber_iu8_moe_tables *>) {
    if ((PyObject *)Py_TYPE(o) != tables_type) return false;
    Py_buffer b;
    if (PyObject_GetBuffer(o, &b, PyBUF_SIMPLE)) return false;
    const bool whole = b.len == (Py_ssize_t)sizeof *v;
    v = (T)b.buf;
    PyBuffer_Release(&b);  // (the structure's own memory: it lives as long as the caller's reference)
    return whole;
  } else if constexpr (std::is_floating_point_v<T>) {
    if (!PyFloat_CheckExact(o)) return false;
    v = (T)PyFloat_AS_DOUBLE(o);
  } else {
    if constexpr (std::is_pointer_v<T>) {
      if (o == Py_None) {
        v = nullptr;
        return true;
      }
    }
    if (!PyLong_CheckExact(o)) return false;
    v = (T)PyLong_AsUnsignedLongLongMask(o);
  }
  return true;
}

template <auto F>
struct Entry;
template <class... A, int (*F)(A...)>
struct Entry<F> {
  static inline PyObject *slow = nullptr;  // the ctypes function
  template <size_t... I>
  static PyObject *go(PyObject *const *args, std::index_sequence<I...>) {
    std::tuple<std::remove_const_t<A>...> v;
    if (!(take(args[I], std::get<I>(v)) && ...)) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = F(std::get<I>(v)...);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
  }
  static PyObject *call(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n == (Py_ssize_t)sizeof...(A)) {
      PyObject *r = go(args, std::index_sequence_for<A...>{});
      if (r || PyErr_Occurred()) return r;
    }
    if (!slow) {
      PyErr_SetString(PyExc_TypeError, "an argument that the ctypes function converts, and none is bound");
      return nullptr;
    }
    return PyObject_Vectorcall(slow, args, (size_t)n, nullptr);
  }
};

#define OPERATORS(X)                                                                                                          \
  X(quant) X(quant_rowmajor) X(gemm) X(rowscale) X(linear_prefill_fused) X(gemm_static) X(gemm_pair) X(linear_fused) X(mlp_chain)  \
  X(gate_up_act) X(quant_had) X(silu_mul_quant_had) X(silu_mul_quant_had_lut) X(add_rms_quant_had) X(gdn_norm_quant_had)          \
  X(attn_gate_quant_had) X(attn_gate_quant_had_lut) X(moe_route) X(moe_route_quant) X(moe_grouped) X(moe_quant_rows)              \
  X(moe_silu_mul_quant) X(moe_gate_up_act) X(moe_down_rows) X(moe_combine)

// bind(functions, tables): {name: ctypes function}, the ctypes structure of the routed operators' tables
PyObject *bind(PyObject *, PyObject *args) {
  PyObject *functions, *tables;
  if (!PyArg_ParseTuple(args, "O!O!", &PyDict_Type, &functions, &PyType_Type, &tables)) return nullptr;
  Py_INCREF(tables);
  Py_XSETREF(tables_type, tables);
#define BIND(name)                                                  \
  if (PyObject *f = PyDict_GetItemString(functions, #name)) {       \
    Py_INCREF(f);                                                   \
    Py_XSETREF(Entry<saber_iu8_##name>::slow, f);                   \
  }
  OPERATORS(BIND)
#undef BIND
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
#define METHOD(name) {#name, (PyCFunction)(void (*)())Entry<saber_iu8_##name>::call, METH_FASTCALL, nullptr},
    OPERATORS(METHOD)
#undef METHOD
    {"bind", bind, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fastcall", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fastcall(void) { return PyModule_Create(&module); }
