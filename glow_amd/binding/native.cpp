// CPython binding of the launch entry points that a Python program calls in its
// inner loop. ctypes builds an object for every argument: 2.1 us for Quantize
// (6 arguments), 4.4 us for a pooled lookup (16) and 6.8 us for
// RowwiseQuantizedFullyConnected (23), several times what the HIP launch behind
// them costs the host. Here the argument types are read off the C ABI's own
// declarations and every argument is converted in place: 0.2 / 0.4 / 0.5 us.
//
// Accepted values are those of the ctypes form (capi._vp, _sz, _i32): a pointer
// is None, an address, an object with a `ptr` (DeviceBuffer, Stream, Event) or
// one that lends its memory (a numpy array, a ctypes structure); an integer is
// anything int() takes, wrapped to the parameter's width.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <tuple>
#include <type_traits>
#include <utility>

#include "glow_mi355x.h"

namespace {

PyObject *g_error = nullptr;    // capi.MI355XError, told by set_error()
PyObject *g_ptr_name = nullptr; // interned "ptr"

bool to_address(PyObject *o, void **out) {
  if (o == Py_None) {
    *out = nullptr;
    return true;
  }
  if (!PyLong_Check(o)) {
    if (PyObject_CheckBuffer(o)) {
      // the caller keeps the object alive across the call, as with ctypes
      Py_buffer view;
      if (PyObject_GetBuffer(o, &view, PyBUF_STRIDES) != 0) return false;
      *out = view.buf;
      PyBuffer_Release(&view);
      return true;
    }
    if (PyObject *p = PyObject_GetAttr(o, g_ptr_name)) {
      const bool ok = to_address(p, out);
      Py_DECREF(p);
      return ok;
    }
    PyErr_Clear();
    PyObject *n = PyNumber_Long(o);
    if (!n) return false;
    const bool ok = to_address(n, out);
    Py_DECREF(n);
    return ok;
  }
  const unsigned long long v = PyLong_AsUnsignedLongLongMask(o);
  if (v == ~0ull && PyErr_Occurred()) return false;
  *out = reinterpret_cast<void *>((uintptr_t)v);
  return true;
}

template <typename T> bool convert(PyObject *o, T &out) {
  if constexpr (std::is_pointer_v<T>) {
    void *p = nullptr;
    if (!to_address(o, &p)) return false;
    out = static_cast<T>(p);
    return true;
  } else if constexpr (std::is_floating_point_v<T>) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) return false;
    out = (T)v;
    return true;
  } else {
    unsigned long long v;
    if (PyLong_Check(o)) {
      v = PyLong_AsUnsignedLongLongMask(o);
    } else {
      PyObject *n = PyNumber_Long(o);
      if (!n) return false;
      v = PyLong_AsUnsignedLongLongMask(n);
      Py_DECREF(n);
    }
    if (v == ~0ull && PyErr_Occurred()) return false;
    out = (T)v;
    return true;
  }
}

PyObject *raise_status(int rc) {
  const char *msg = mi355x_last_error();
  if (!g_error) {
    PyErr_Format(PyExc_RuntimeError, "mi355x status %d: %s", rc, msg);
    return nullptr;
  }
  if (PyObject *e = PyObject_CallFunction(g_error, "is", rc, msg)) {
    PyErr_SetObject(g_error, e);
    Py_DECREF(e);
  }
  return nullptr;
}

// One entry point int fn(Args...): converts, calls without the interpreter lock
// (a launch may wait for room in the queue), raises on a status other than 0.
template <auto Fn> struct Entry;
template <typename... Args, int (*Fn)(Args...)> struct Entry<Fn> {
  template <size_t... I>
  static PyObject *call(PyObject *const *a, std::index_sequence<I...>) {
    std::tuple<Args...> v;
    if (!(convert(a[I], std::get<I>(v)) && ...)) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = Fn(std::get<I>(v)...);
    Py_END_ALLOW_THREADS
    if (rc != MI355X_OK) return raise_status(rc);
    Py_RETURN_NONE;
  }
  static PyObject *fast(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != (Py_ssize_t)sizeof...(Args))
      return PyErr_Format(PyExc_TypeError, "%zd arguments given, %zu expected", n, sizeof...(Args));
    return call(args, std::index_sequence_for<Args...>{});
  }
};

PyObject *set_error(PyObject *, PyObject *cls) {
  Py_INCREF(cls);
  Py_XSETREF(g_error, cls);
  Py_RETURN_NONE;
}

#define ENTRY(name)                                                                              \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Entry<&mi355x_##name>::fast)), \
   METH_FASTCALL, nullptr}

PyMethodDef g_methods[] = {
    {"set_error", set_error, METH_O, nullptr},
    ENTRY(quantize_i8),
    ENTRY(dequantize_i8),
    ENTRY(rescale_i8),
    ENTRY(copy_u8),
    ENTRY(rowsum_i8),
    ENTRY(add_i8),
    ENTRY(add_relu_i8),
    ENTRY(rwq_fc_i8),
    ENTRY(rwq_fc_i8_opts),
    ENTRY(cwq_conv2d_i8),
    ENTRY(cwq_conv2d_i8_opts),
    ENTRY(cwq_conv2d_add_i8),
    ENTRY(frwq_slws),
    ENTRY(frwq_slws_opts),
    ENTRY(frwq_slws_noalloc),
    ENTRY(frwq_slws_noalloc_opts),
    ENTRY(frwq_slws_offsets),
    ENTRY(frwq_slws_offsets_opts),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, g_methods,
                        nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__native(void) {
  g_ptr_name = PyUnicode_InternFromString("ptr");
  return g_ptr_name ? PyModule_Create(&g_module) : nullptr;
}
