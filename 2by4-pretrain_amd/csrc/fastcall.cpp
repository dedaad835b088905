// The C ABI of tf24.h as functions of a CPython module, for the calls that sit on the host path of every product and step.
//
// ctypes converts each argument through a Python object of its own: 1.5 us for 10 arguments, 2.4 for the 20 of tf24_spmm, of the 11 us that
// torch.nn.functional.linear with a 2:4 weight takes.  Here the argument types come from the declarations in tf24.h, and a call takes what
// its conversions do.  As with ctypes a pointer is an address, bytes, None or an object of ctypes, an integer is taken modulo the size of its type,
// and other Python threads run while the call does.  Only the stable ABI is used: one binary for every CPython from 3.10 on.
#define PY_SSIZE_T_CLEAN
#define Py_LIMITED_API 0x030a0000
#include <Python.h>
#include <cstdint>
#include <tuple>
#include <type_traits>
#include <utility>
#include "tf24.h"

namespace {

// address that an object of ctypes (a pointer, an array, byref(..)) stands for
bool ctypes_address(PyObject* o, void*& out) {
  PyObject *ctypes = nullptr, *type = nullptr, *cast = nullptr, *value = nullptr;
  if (!PyUnicode_Check(o) && (ctypes = PyImport_ImportModule("ctypes")) && (type = PyObject_GetAttrString(ctypes, "c_void_p")) &&
      (cast = PyObject_CallMethod(ctypes, "cast", "OO", o, type)))
    value = PyObject_GetAttrString(cast, "value");
  const bool ok = value && (value == Py_None || PyLong_Check(value));
  if (ok) out = value == Py_None ? nullptr : (void*)(uintptr_t)PyLong_AsUnsignedLongLongMask(value);
  Py_XDECREF(value); Py_XDECREF(cast); Py_XDECREF(type); Py_XDECREF(ctypes);
  if (!ok) PyErr_SetString(PyExc_TypeError, "a pointer is given as an address, bytes, None or an object of ctypes");
  return ok;
}

template <typename T>
bool number(PyObject* o, T& out) {
  if constexpr (std::is_floating_point_v<T>) out = (T)PyFloat_AsDouble(o);
  else out = (T)PyLong_AsUnsignedLongLongMask(o);                // (a float has no __index__: TypeError)
  return out != (T)-1 || !PyErr_Occurred();                      // (either returns -1 with an error)
}

template <typename T>
bool from_object(PyObject* o, T& out) {
  if constexpr (std::is_pointer_v<T>) {
    void* at = nullptr;
    if (o == Py_None) at = nullptr;
    else if (PyLong_Check(o)) at = (void*)(uintptr_t)PyLong_AsUnsignedLongLongMask(o);
    else if (PyBytes_Check(o)) at = PyBytes_AsString(o);         // (held by the caller's arguments)
    else if (!ctypes_address(o, at)) return false;
    out = (T)at;
    return true;
  } else {
    static_assert(std::is_floating_point_v<T> || std::is_integral_v<T>, "tf24.h passes pointers, floating-point numbers and integers");
    if (number(o, out)) return true;
    PyObject *type, *error, *trace;                              // a number of ctypes holds it as its `value`
    PyErr_Fetch(&type, &error, &trace);
    PyObject* value = PyObject_HasAttrString(o, "_type_") ? PyObject_GetAttrString(o, "value") : nullptr;
    PyErr_Clear();
    const bool ok = value && number(value, out);
    Py_XDECREF(value);
    if (ok || PyErr_Occurred()) { Py_XDECREF(type); Py_XDECREF(error); Py_XDECREF(trace); }
    else PyErr_Restore(type, error, trace);
    return ok;
  }
}

template <auto FN, typename R, typename... A, size_t... I>
PyObject* call_with(R (*)(A...), PyObject* const* args, std::index_sequence<I...>) {
  std::tuple<std::remove_cv_t<A>...> v;
  if (!(from_object(args[I], std::get<I>(v)) && ...)) return nullptr;
  R r;
  Py_BEGIN_ALLOW_THREADS
  r = FN(std::get<I>(v)...);
  Py_END_ALLOW_THREADS
  return PyLong_FromLongLong((long long)r);
}
template <typename R, typename... A>
constexpr size_t arity(R (*)(A...)) { return sizeof...(A); }
template <auto FN>
PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
  constexpr size_t N = arity(FN);
  if (n != (Py_ssize_t)N) { PyErr_Format(PyExc_TypeError, "%zd arguments given, %zu expected", n, N); return nullptr; }
  return call_with<FN>(FN, args, std::make_index_sequence<N>{});
}

#define TF24_METHOD(name) {#name, (PyCFunction)(void (*)(void))call<&name>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    TF24_METHOD(tf24_prune_compress), TF24_METHOD(tf24_prune_compress_rowsum), TF24_METHOD(tf24_prune_compress_rowsum_workspace_bytes),
    TF24_METHOD(tf24_prune_compress_dual), TF24_METHOD(tf24_decompress), TF24_METHOD(tf24_repack_to), TF24_METHOD(tf24_transposable_mask),
    TF24_METHOD(tf24_soft_threshold24), TF24_METHOD(tf24_soft_threshold24_scaled), TF24_METHOD(tf24_soft_threshold24_scaled_bias),
    TF24_METHOD(tf24_masked_add), TF24_METHOD(tf24_adamw_masked_decay_list), TF24_METHOD(tf24_gelu_glu_forward), TF24_METHOD(tf24_gelu_glu_backward),
    TF24_METHOD(tf24_spmm), TF24_METHOD(tf24_linear), TF24_METHOD(tf24_spmm_workspace_bytes), TF24_METHOD(tf24_grad_weight), TF24_METHOD(tf24_grad_weight_f32),
    TF24_METHOD(tf24_grad_weight_workspace_bytes), TF24_METHOD(tf24_linear16), TF24_METHOD(tf24_linear16_suits), TF24_METHOD(tf24_transpose),
    TF24_METHOD(tf24_mvue_weight_grad), TF24_METHOD(tf24_mvue_weight_grad_workspace_bytes),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fastcall", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fastcall() { return PyModule_Create(&module); }
