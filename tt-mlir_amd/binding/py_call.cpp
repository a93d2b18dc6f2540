// The kernel library's entry points as Python calls: what hip.call() and hip.ptr() do, with the argument types known at compile time.
// A call through ctypes converts each argument by a look-up and an object of its own and took 1.1 (8 arguments) to 2.1 us (18), a
// device address 0.5 us: more than a small kernel.  Only ints, floats, None and ctypes.c_void_p objects are converted here; a
// call with anything else in it (byref, arrays, bytes, keywords, a wrong number of arguments) goes to the ctypes function as it is, and so does every
// call while buffer extents are checked.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstddef>
#include <cstdint>
#include <tuple>
#include <type_traits>
#include <utility>

#include "ttmlir_amd_hip.h"

namespace {

PyTypeObject *voidPointer = nullptr;   // ctypes.c_void_p
PyObject *addressType = nullptr, *slowCall = nullptr, *slowPtr = nullptr, *raiseStatus = nullptr;   // hip.py's
PyObject *entries = nullptr;           // {name: capsule of an Entry}
PyObject *sContiguous, *sDataPtr, *sBytes;
bool checking = false;

// Python value -> C argument with ctypes' conversions (integers lose their upper bits); false: not one of the plain types
template <class T>
bool take(PyObject *o, T &v) {
  if constexpr (std::is_pointer_v<T>) {
    if (o == Py_None) {
      v = nullptr;
      return true;
    }
    if (PyLong_Check(o)) {
      v = reinterpret_cast<T>(static_cast<std::uintptr_t>(PyLong_AsUnsignedLongLongMask(o)));
      return true;
    }
    if (!PyObject_TypeCheck(o, voidPointer)) return false;
    Py_buffer b;
    if (PyObject_GetBuffer(o, &b, PyBUF_SIMPLE) != 0) {
      PyErr_Clear();
      return false;
    }
    const bool whole = b.len == static_cast<Py_ssize_t>(sizeof(void *));
    if (whole) v = *static_cast<T *>(b.buf);
    PyBuffer_Release(&b);
    return whole;
  } else if constexpr (std::is_floating_point_v<T>) {
    if (PyFloat_Check(o)) {
      v = static_cast<T>(PyFloat_AS_DOUBLE(o));
      return true;
    }
    if (!PyLong_Check(o)) return false;
    const double d = PyLong_AsDouble(o);
    if (d == -1.0 && PyErr_Occurred()) {
      PyErr_Clear();
      return false;
    }
    v = static_cast<T>(d);
    return true;
  } else {
    if (!PyLong_Check(o)) return false;
    v = static_cast<T>(PyLong_AsUnsignedLongLongMask(o));
    return true;
  }
}

template <class T>
constexpr bool plain = std::is_arithmetic_v<T> || (std::is_pointer_v<T> && !std::is_same_v<T, const char *> && !std::is_same_v<T, char *>);

struct Entry {
  void *fn = nullptr;
  Py_ssize_t count = 0;
  bool (*invoke)(void *fn, PyObject *const *args, int &status) = nullptr;
};

template <class... A, std::size_t... I>
bool invokeAs(void *fn, PyObject *const *args, int &status, std::index_sequence<I...>) {
  std::tuple<A...> v;
  if (!(take(args[I], std::get<I>(v)) && ...)) return false;
  Py_BEGIN_ALLOW_THREADS   // some of them wait for the device
  status = reinterpret_cast<int (*)(A...)>(fn)(std::get<I>(v)...);
  Py_END_ALLOW_THREADS
  return true;
}
template <class... A>
Entry entryFor(int (*)(A...)) {
  Entry e;
  e.count = sizeof...(A);
  if constexpr ((plain<A> && ...))
    e.invoke = [](void *fn, PyObject *const *args, int &status) { return invokeAs<A...>(fn, args, status, std::index_sequence_for<A...>{}); };
  return e;
}
template <class R, class... A>
Entry entryFor(R (*)(A...)) {   // no status to check: left to ctypes
  return {};
}

struct Named {
  const char *name;
  Entry entry;
};
Named table[] = {
#define TTM_ENTRY(name) {#name, entryFor(static_cast<decltype(&name)>(nullptr))},
#include "ttm_entries.inc"
#undef TTM_ENTRY
};

PyObject *names(PyObject *, PyObject *) {
  PyObject *l = PyList_New(0);
  for (const Named &n : table) {
    PyObject *s = l && n.entry.invoke ? PyUnicode_FromString(n.name) : nullptr;
    if (s && PyList_Append(l, s) != 0) Py_CLEAR(l);
    Py_XDECREF(s);
  }
  return l;
}

// bind({name: address}): the functions that calls go to from now on
PyObject *bind(PyObject *, PyObject *addresses) {
  PyObject *fresh = PyDict_New();
  if (!fresh) return nullptr;
  for (Named &n : table) {
    PyObject *a = PyDict_Check(addresses) ? PyDict_GetItemString(addresses, n.name) : nullptr;
    if (!a || !n.entry.invoke) continue;
    n.entry.fn = PyLong_AsVoidPtr(a);
    PyObject *c = n.entry.fn ? PyCapsule_New(&n.entry, nullptr, nullptr) : nullptr;
    if (!c || PyDict_SetItemString(fresh, n.name, c) != 0) {
      Py_XDECREF(c);
      Py_DECREF(fresh);
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: a null address");
      return nullptr;
    }
    Py_DECREF(c);
  }
  Py_XSETREF(entries, fresh);
  Py_RETURN_NONE;
}

// setup(c_void_p, address type, call, ptr, check)
PyObject *setup(PyObject *, PyObject *args) {
  PyObject *vp, *at, *sc, *sp, *rs;
  if (!PyArg_ParseTuple(args, "O!OOOO", &PyType_Type, &vp, &at, &sc, &sp, &rs)) return nullptr;
  for (PyObject *o : {vp, at, sc, sp, rs}) Py_INCREF(o);   // for good: the module lives as long as the process
  voidPointer = reinterpret_cast<PyTypeObject *>(vp);
  addressType = at; slowCall = sc; slowPtr = sp; raiseStatus = rs;
  Py_RETURN_NONE;
}

PyObject *check(PyObject *, PyObject *on) {
  const int v = PyObject_IsTrue(on);
  if (v < 0) return nullptr;
  checking = v != 0;
  Py_RETURN_NONE;
}

PyObject *call(PyObject *, PyObject *const *args, Py_ssize_t n, PyObject *keywords) {
  if (!slowCall) {
    PyErr_SetString(PyExc_RuntimeError, "call before setup");
    return nullptr;
  }
  if (n < 1 || keywords || checking) return PyObject_Vectorcall(slowCall, args, static_cast<size_t>(n), keywords);
  PyObject *c = entries ? PyDict_GetItemWithError(entries, args[0]) : nullptr;
  if (!c && PyErr_Occurred()) PyErr_Clear();
  const Entry *e = c ? static_cast<const Entry *>(PyCapsule_GetPointer(c, nullptr)) : nullptr;
  int status = 0;
  if (!e || n - 1 != e->count || !e->invoke(e->fn, args + 1, status)) return PyObject_Vectorcall(slowCall, args, static_cast<size_t>(n), nullptr);
  if (status != 0) {
    PyObject *s = PyLong_FromLong(status);
    PyObject *r = s ? PyObject_CallFunctionObjArgs(raiseStatus, s, args[0], nullptr) : nullptr;
    Py_XDECREF(s);
    return r;
  }
  Py_RETURN_NONE;
}

PyObject *ptr(PyObject *, PyObject *const *args, Py_ssize_t n_args, PyObject *keywords) {
  if (!slowPtr) {
    PyErr_SetString(PyExc_RuntimeError, "ptr before setup");
    return nullptr;
  }
  if (n_args != 1 || keywords) return PyObject_Vectorcall(slowPtr, args, static_cast<size_t>(n_args), keywords);
  PyObject *t = args[0];
  PyObject *dense = PyObject_CallMethodNoArgs(t, sContiguous);
  if (!dense) return nullptr;
  const bool yes = dense == Py_True;
  Py_DECREF(dense);
  if (!yes) return PyObject_CallOneArg(slowPtr, t);   // says what is wrong
  PyObject *a = PyObject_CallMethodNoArgs(t, sDataPtr), *p = a ? PyObject_CallOneArg(addressType, a) : nullptr;
  Py_XDECREF(a);
  PyObject *n = p ? PyObject_GetAttr(t, sBytes) : nullptr;
  if (!n || PyObject_SetAttr(p, sBytes, n) != 0) Py_CLEAR(p);
  Py_XDECREF(n);
  return p;
}

PyMethodDef methods[] = {
    {"setup", setup, METH_VARARGS, nullptr},
    {"names", names, METH_NOARGS, "The entry points that can be bound."},
    {"bind", bind, METH_O, nullptr},
    {"check", check, METH_O, nullptr},
    {"call", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(call)), METH_FASTCALL | METH_KEYWORDS,
     "call(name, *args): the entry point `name` of the kernel library; raises TTMError if it fails."},
    {"ptr", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(ptr)), METH_FASTCALL | METH_KEYWORDS,
     "Device address of a torch tensor (must be contiguous); it carries the tensor's size for check_buffers."},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ttm_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ttm_call() {
  sContiguous = PyUnicode_InternFromString("is_contiguous");
  sDataPtr = PyUnicode_InternFromString("data_ptr");
  sBytes = PyUnicode_InternFromString("nbytes");
  return sContiguous && sDataPtr && sBytes ? PyModule_Create(&module) : nullptr;
}
