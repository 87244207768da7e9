// it_pycall.cpp -- CPython bindings of the entry points a serving loop calls
// on every step (module infer_train_amd._call).
//
// ctypes converts each argument through Python-level descriptors: an 18-
// argument call costs ~3 us before the library sees it, more than a kernel
// launch.  Here the C signature of each function (include/it_kv.h) drives the
// conversion at compile time, for the arguments a call nearly always has: ints
// (masked to the parameter's width), ints or None for pointers, floats or ints
// for floats.  A call with any other argument is handed to the ctypes function
// as it is, so what ctypes takes (__index__, ctypes instances, _as_parameter_)
// is taken and what it refuses is refused with its error (and a str, which
// c_void_p would take for the address of its characters).  Only
// it_paged_decode_partition takes more: its arrays are host memory and may be
// given as buffers.  The GIL is released around the call, as ctypes does.
//
// The functions are looked up in the library that the package has loaded
// (bind(path, lib)), not linked.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <dlfcn.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "it_kv.h"

namespace {
PyObject* argument_error = nullptr;  // ctypes.ArgumentError

// The value of an argument that needs no more than this; false: ctypes decides.
// kHost: the function's pointers are host memory, given as addresses or as
// buffers (const: of one dimension or more; else writable).
template <bool kHost, class T>
bool convert(PyObject* o, T& v) {
  if constexpr (std::is_floating_point_v<T>) {
    if (!PyFloat_Check(o) && !PyLong_Check(o)) return false;
    const double d = PyFloat_AsDouble(o);  // an int past the double range fails
    if (d == -1.0 && PyErr_Occurred()) {
      PyErr_Clear();
      return false;
    }
    v = static_cast<T>(d);
  } else if (PyLong_Check(o)) {
    const unsigned long long x = PyLong_AsUnsignedLongLongMask(o);
    if constexpr (std::is_pointer_v<T>) v = reinterpret_cast<T>(static_cast<uintptr_t>(x));
    else v = static_cast<T>(x);
  } else if constexpr (std::is_pointer_v<T>) {
    v = T{};
    if (o == Py_None) return true;
    if (!kHost || !PyObject_CheckBuffer(o)) return false;
    constexpr bool kConst = std::is_const_v<std::remove_pointer_t<T>>;
    Py_buffer b;
    if (PyObject_GetBuffer(o, &b, kConst ? PyBUF_ND : PyBUF_ND | PyBUF_WRITABLE)) {
      PyErr_Clear();
      return false;
    }
    const bool taken = !kConst || b.ndim > 0;
    v = reinterpret_cast<T>(b.buf);  // the caller keeps the object for the call
    PyBuffer_Release(&b);
    return taken;
  } else {
    return false;
  }
  return true;
}

template <bool kHost, class F>
struct Call;
template <bool kHost, class R, class... A>
struct Call<kHost, R (*)(A...)> {
  using Fn = R (*)(A...);
  template <size_t... I>
  static PyObject* run(Fn f, PyObject* ctypes, PyObject* const* args, Py_ssize_t n, std::index_sequence<I...>) {
    std::tuple<A...> v{};
    if (n != Py_ssize_t(sizeof...(A)) || !(convert<kHost>(args[I], std::get<I>(v)) && ...)) {
      for (Py_ssize_t i = 0; i < n; ++i)
        if (PyUnicode_Check(args[i])) return PyErr_Format(argument_error, "argument %zd: a str is not an address", i + 1);
      return PyObject_Vectorcall(ctypes, args, size_t(n), nullptr);
    }
    R r;
    Py_BEGIN_ALLOW_THREADS r = f(std::get<I>(v)...);
    Py_END_ALLOW_THREADS
    if constexpr (std::is_signed_v<R>) return PyLong_FromLongLong(r);
    else return PyLong_FromUnsignedLongLong(r);
  }
  static PyObject* run(const char* name, Fn f, PyObject* ctypes, PyObject* const* args, Py_ssize_t n) {
    if (!f) {
      PyErr_Format(PyExc_RuntimeError, "%s: bind() the library first", name);
      return nullptr;
    }
    return run(f, ctypes, args, n, std::index_sequence_for<A...>{});
  }
};

#define IT_CALLS(X)                                                                                                      \
  X(it_kv_append, false) X(it_kv_append_rope, false) X(it_kv_gather, false) X(it_kv_evict, false)                        \
  X(it_kv_sync_tables, false) X(it_kv_copy_blocks, false) X(it_paged_decode_workspace, false)                            \
  X(it_paged_decode_partition, true) X(it_paged_decode, false) X(it_paged_decode_split, false)                           \
  X(it_paged_decode_combine, false) X(it_paged_prefill_workspace, false) X(it_paged_prefill_ws, false)                   \
  X(it_flash_attention_workspace, false) X(it_flash_attention, false)

#define IT_WRAP(name, host)                                                         \
  decltype(&name) p_##name = nullptr;                                               \
  PyObject* c_##name = nullptr;                                                     \
  PyObject* py_##name(PyObject*, PyObject* const* args, Py_ssize_t n) {             \
    return Call<host, decltype(&name)>::run(#name, p_##name, c_##name, args, n);    \
  }
IT_CALLS(IT_WRAP)

PyObject* bind(PyObject*, PyObject* args) {
  const char* path;
  PyObject* table;
  if (!PyArg_ParseTuple(args, "sO", &path, &table)) return nullptr;
  void* lib = dlopen(path, RTLD_NOW | RTLD_NOLOAD);
  if (!lib) return PyErr_Format(PyExc_ImportError, "%s is not loaded", path);
#define IT_BIND(name, host)                                                                                       \
  Py_XSETREF(c_##name, PyObject_GetAttrString(table, #name));                                                     \
  if (!c_##name) return nullptr;                                                                                  \
  p_##name = reinterpret_cast<decltype(p_##name)>(dlsym(lib, #name));                                             \
  if (!p_##name) return PyErr_Format(PyExc_ImportError, "%s does not export " #name, path);
  IT_CALLS(IT_BIND)
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, "bind(path, lib): the entry points of the loaded library at this path, lib its ctypes table."},
#define IT_METHOD(name, host) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_##name)), METH_FASTCALL, nullptr},
    IT_CALLS(IT_METHOD){nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_call", "Bindings of include/it_kv.h's per-step entry points.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};
}  // namespace

PyMODINIT_FUNC PyInit__call() {
  PyObject* const ctypes = PyImport_ImportModule("ctypes");
  if (!ctypes) return nullptr;
  argument_error = PyObject_GetAttrString(ctypes, "ArgumentError");
  Py_DECREF(ctypes);
  return argument_error ? PyModule_Create(&module) : nullptr;
}
