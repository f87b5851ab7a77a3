// The interpreter's way to the kernel libraries' entry points: one builtin function per entry point, which checks the number of
// its arguments, turns them into the entry point's types and calls it without the interpreter's lock.
// bind(name, address) -> builtin.  The table of entry points and their types is made from ops/signatures.py by the build.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstring>
#include <tuple>
#include <utility>

namespace {

// None is a null pointer, whole numbers wrap as they do in C, and any number is a float
template <typename T> inline T argument(PyObject* o) { return static_cast<T>(PyLong_AsUnsignedLongLongMask(o)); }
template <> inline void* argument<void*>(PyObject* o) { return o == Py_None ? nullptr : reinterpret_cast<void*>(PyLong_AsUnsignedLongLongMask(o)); }
template <> inline float argument<float>(PyObject* o) { return static_cast<float>(PyFloat_AsDouble(o)); }
template <> inline double argument<double>(PyObject* o) { return PyFloat_AsDouble(o); }

template <int ID, typename... A>
struct Entry {
  static int (*function)(A...);

  template <size_t... N>
  static PyObject* run(PyObject* const* args, std::index_sequence<N...>) {
    const std::tuple<A...> values{argument<A>(args[N])...};
    if (PyErr_Occurred()) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = std::apply(function, values);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
  }

  static PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t count) {
    if (count != static_cast<Py_ssize_t>(sizeof...(A))) {
      PyErr_Format(PyExc_TypeError, "entry point takes %zd arguments, got %zd", static_cast<Py_ssize_t>(sizeof...(A)), count);
      return nullptr;
    }
    return run(args, std::index_sequence_for<A...>{});
  }

  static void bind(void* address) { function = reinterpret_cast<int (*)(A...)>(address); }
};
template <int ID, typename... A> int (*Entry<ID, A...>::function)(A...) = nullptr;

struct Known {
  PyMethodDef method;
  void (*bind)(void*);
};

#define ENTRY(id, name, ...) \
  {{#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Entry<id, __VA_ARGS__>::call)), METH_FASTCALL, nullptr}, &Entry<id, __VA_ARGS__>::bind},
Known known[] = {
#include "launch_entries.inc"
};
#undef ENTRY

PyObject* bind(PyObject*, PyObject* args) {
  const char* name;
  PyObject* address;
  if (!PyArg_ParseTuple(args, "sO", &name, &address)) return nullptr;
  void* p = PyLong_AsVoidPtr(address);
  if (!p) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "an entry point without an address");
    return nullptr;
  }
  for (Known& k : known)
    if (!std::strcmp(k.method.ml_name, name)) {
      k.bind(p);
      return PyCFunction_New(&k.method, nullptr);
    }
  PyErr_Format(PyExc_KeyError, "no entry point %s", name);
  return nullptr;
}

PyMethodDef functions[] = {{"bind", bind, METH_VARARGS, "bind(name, address): the entry point as a builtin function"}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_definition = {PyModuleDef_HEAD_INIT, "photon_launch", nullptr, -1, functions, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_photon_launch(void) { return PyModule_Create(&module_definition); }
