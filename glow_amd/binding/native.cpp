// CPython binding of the entry points that a Python program calls in its inner
// loop: the launches, and requests to a device manager. ctypes builds an object for
// every argument: 2.1 us for Quantize (6 arguments), 4.4 us for a pooled lookup (16)
// and 6.8 us for RowwiseQuantizedFullyConnected (23), several times what the HIP
// launch behind them costs the host. Here the argument types are read off the C ABI's
// own declarations and every argument is converted in place: 0.2 / 0.4 / 0.5 us.
//
// A pointer is None, an address (anything int() takes, numpy's integers among them), an
// object with a `ptr` (DeviceBuffer, Stream, Event), or the memory of an object of the
// types told by set_memory_types() (numpy arrays, ctypes structures and arrays). Other
// objects that lend their memory, a numpy or ctypes scalar for one, are not taken for
// it. An integer is anything int() takes, wrapped to the parameter's width.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <tuple>
#include <type_traits>
#include <utility>
#include <vector>

#include "glow_mi355x.h"
#include "glow_mi355x_host.h"

namespace {

PyObject *g_error = nullptr;    // capi.MI355XError, told by set_error()
PyObject *g_host_error = nullptr; // host.HostError
PyObject *g_ptr_name = nullptr; // interned "ptr"
PyObject *g_memory = nullptr;   // tuple of types whose instances stand for their memory

bool is_memory(PyObject *o) {
  // (isinstance() asks every type's metaclass: 0.1 us an argument)
  for (Py_ssize_t i = 0; g_memory && i < PyTuple_GET_SIZE(g_memory); i++)
    if (PyType_IsSubtype(Py_TYPE(o), reinterpret_cast<PyTypeObject *>(PyTuple_GET_ITEM(g_memory, i))))
      return true;
  return false;
}

bool to_address(PyObject *o, void **out) {
  if (o == Py_None) {
    *out = nullptr;
    return true;
  }
  if (!PyLong_Check(o)) {
    if (is_memory(o)) {
      // the caller keeps the object alive across the call, as with ctypes
      Py_buffer view;
      if (PyObject_GetBuffer(o, &view, PyBUF_STRIDES) != 0) return false;
      *out = view.buf;
      PyBuffer_Release(&view);
      return true;
    }
    PyObject *p = PyObject_GetAttr(o, g_ptr_name);
    if (!p) {
      PyErr_Clear();
      p = PyNumber_Long(o);
      if (!p) return false;
    }
    const bool ok = to_address(p, out);
    Py_DECREF(p);
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

PyObject *set_memory_types(PyObject *, PyObject *types) {
  if (!PyTuple_Check(types)) return PyErr_Format(PyExc_TypeError, "a tuple of types is expected");
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(types); i++)
    if (!PyType_Check(PyTuple_GET_ITEM(types, i)))
      return PyErr_Format(PyExc_TypeError, "a tuple of types is expected");
  Py_INCREF(types);
  Py_XSETREF(g_memory, types);
  Py_RETURN_NONE;
}

PyObject *set_host_error(PyObject *, PyObject *cls) {
  Py_INCREF(cls);
  Py_XSETREF(g_host_error, cls);
  Py_RETURN_NONE;
}

// dm_run(handle, function name, {placeholder name: array}): a request, without the
// ctypes arrays of names, addresses and sizes (45 us for the 57 bindings of a
// ranking request).
PyObject *dm_run(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  if (nargs != 3) return PyErr_Format(PyExc_TypeError, "%zd arguments given, 3 expected", nargs);
  void *dm = nullptr;
  if (!to_address(args[0], &dm)) return nullptr;
  const char *name = PyUnicode_AsUTF8(args[1]);
  if (!name) return nullptr;
  if (!PyDict_Check(args[2])) return PyErr_Format(PyExc_TypeError, "bindings are a dict");
  const size_t n = (size_t)PyDict_Size(args[2]);
  std::vector<const char *> names;
  std::vector<void *> data;
  std::vector<size_t> bytes;
  std::vector<Py_buffer> views;    // held while the request runs
  names.reserve(n), data.reserve(n), bytes.reserve(n), views.reserve(n);
  PyObject *key, *value;
  Py_ssize_t pos = 0;
  bool ok = true;
  while (ok && PyDict_Next(args[2], &pos, &key, &value)) {
    const char *k = PyUnicode_AsUTF8(key);
    Py_buffer view;
    ok = k && PyObject_GetBuffer(value, &view, PyBUF_STRIDES) == 0;
    if (!ok) break;
    views.push_back(view);
    ok = PyBuffer_IsContiguous(&view, 'C');
    if (!ok) {
      PyErr_Format(PyExc_AssertionError, "the array bound to %s is not C-contiguous", k);
      break;
    }
    names.push_back(k);
    data.push_back(view.buf);
    bytes.push_back((size_t)view.len);
  }
  int rc = 0;
  if (ok) {
    Py_BEGIN_ALLOW_THREADS
    rc = mi355x_host_dm_run(static_cast<mi355x_host_dm *>(dm), name, names.data(), data.data(),
                            bytes.data(), (int)names.size());
    Py_END_ALLOW_THREADS
  }
  for (Py_buffer &v : views) PyBuffer_Release(&v);
  if (!ok) return nullptr;
  if (rc < 0) {
    const char *msg = mi355x_host_last_error();
    if (!g_host_error) return PyErr_Format(PyExc_RuntimeError, "status %d: %s", -rc, msg);
    if (PyObject *e = PyObject_CallFunction(g_host_error, "is", -rc, msg)) {
      PyErr_SetObject(g_host_error, e);
      Py_DECREF(e);
    }
    return nullptr;
  }
  Py_RETURN_NONE;
}

#define ENTRY(name)                                                                              \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Entry<&mi355x_##name>::fast)), \
   METH_FASTCALL, nullptr}

PyMethodDef g_methods[] = {
    {"set_error", set_error, METH_O, nullptr},
    {"set_memory_types", set_memory_types, METH_O, nullptr},
    {"set_host_error", set_host_error, METH_O, nullptr},
    {"dm_run", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&dm_run)), METH_FASTCALL,
     nullptr},
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
