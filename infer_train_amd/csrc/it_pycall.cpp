// it_pycall.cpp -- CPython bindings of the entry points a serving loop calls
// on every step (module infer_train_amd._call).
//
// ctypes converts each argument through Python-level descriptors: an 18-
// argument call costs ~3 us before the library sees it, more than a kernel
// launch.  Here the C signature of each function (include/it_kv.h) drives the
// conversion at compile time.  Arguments are what the ctypes table takes:
// integers (masked to the parameter's width), addresses, None or host buffers
// for pointers, and floats; the result is the function's integer.  The GIL is released
// around the call, as ctypes does.
//
// The functions are looked up in the library that the package has loaded
// (bind(path)), not linked.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <dlfcn.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "it_kv.h"

namespace {
PyObject* argument_error = nullptr;  // ctypes.ArgumentError: what the ctypes table raises

// An int for an integer; an int, None or an object with a contiguous buffer
// for a pointer; a number for a float.  Anything else is refused.
template <class T>
T convert(PyObject* o) {
  if constexpr (std::is_floating_point_v<T>) {
    return static_cast<T>(PyFloat_AsDouble(o));
  } else if (PyLong_Check(o)) {
    if constexpr (std::is_pointer_v<T>) return reinterpret_cast<T>(PyLong_AsVoidPtr(o));
    else return static_cast<T>(PyLong_AsUnsignedLongLongMask(o));
  } else if (std::is_pointer_v<T> && o == Py_None) {
    return T{};
  } else if (std::is_pointer_v<T> && PyObject_CheckBuffer(o)) {
    // Host memory (a numpy array, a ctypes value); the caller keeps it.
    Py_buffer b;
    if (PyObject_GetBuffer(o, &b, PyBUF_SIMPLE)) return T{};
    void* const p = b.buf;
    PyBuffer_Release(&b);
    if constexpr (std::is_pointer_v<T>) return reinterpret_cast<T>(p);
  } else {
    PyErr_Format(argument_error, "int expected instead of %s instance", Py_TYPE(o)->tp_name);
  }
  return T{};
}

template <class F>
struct Call;
template <class R, class... A>
struct Call<R (*)(A...)> {
  using Fn = R (*)(A...);
  template <size_t... I>
  static PyObject* run(Fn f, PyObject* const* args, std::index_sequence<I...>) {
    std::tuple<A...> v{convert<A>(args[I])...};  // braces: converted in order
    if (PyErr_Occurred()) return nullptr;
    R r;
    Py_BEGIN_ALLOW_THREADS r = f(std::get<I>(v)...);
    Py_END_ALLOW_THREADS
    if constexpr (std::is_signed_v<R>) return PyLong_FromLongLong(r);
    else return PyLong_FromUnsignedLongLong(r);
  }
  static PyObject* run(const char* name, Fn f, PyObject* const* args, Py_ssize_t n) {
    if (!f) {
      PyErr_Format(PyExc_RuntimeError, "%s: bind() the library first", name);
      return nullptr;
    }
    if (n != Py_ssize_t(sizeof...(A))) {
      PyErr_Format(PyExc_TypeError, "%s takes %zd arguments (%zd given)", name, Py_ssize_t(sizeof...(A)), n);
      return nullptr;
    }
    return run(f, args, std::index_sequence_for<A...>{});
  }
};

#define IT_CALLS(X)                                                                                        \
  X(it_kv_append) X(it_kv_append_rope) X(it_kv_gather) X(it_kv_evict) X(it_kv_sync_tables)                 \
  X(it_kv_copy_blocks) X(it_paged_decode_workspace) X(it_paged_decode_partition) X(it_paged_decode)        \
  X(it_paged_decode_split) X(it_paged_decode_combine) X(it_paged_prefill_workspace) X(it_paged_prefill_ws) \
  X(it_flash_attention_workspace) X(it_flash_attention)

#define IT_WRAP(name)                                                               \
  decltype(&name) p_##name = nullptr;                                               \
  PyObject* py_##name(PyObject*, PyObject* const* args, Py_ssize_t n) {             \
    return Call<decltype(&name)>::run(#name, p_##name, args, n);                    \
  }
IT_CALLS(IT_WRAP)

PyObject* bind(PyObject*, PyObject* arg) {
  const char* path = PyUnicode_AsUTF8(arg);
  if (!path) return nullptr;
  void* lib = dlopen(path, RTLD_NOW | RTLD_NOLOAD);
  if (!lib) return PyErr_Format(PyExc_ImportError, "%s is not loaded", path);
#define IT_BIND(name)                                                                                             \
  p_##name = reinterpret_cast<decltype(p_##name)>(dlsym(lib, #name));                                             \
  if (!p_##name) return PyErr_Format(PyExc_ImportError, "%s does not export " #name, path);
  IT_CALLS(IT_BIND)
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", bind, METH_O, "Look the entry points up in the loaded library at this path."},
#define IT_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_##name)), METH_FASTCALL, nullptr},
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
