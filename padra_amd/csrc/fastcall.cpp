// The Python front end's way into libpadra_hip.so: one function per entry point, with the
// C-ABI's arguments after the tensor whose device and current stream the call runs on.  A
// device pointer is a tensor (or None), a descriptor its own ctypes structure (or None).
//
// A decode step's kernels take 3-5 us, and ctypes with its Python-side conversions took 8-16 us a
// call, so the calls and not the kernels set the time of every small launch.  These read the
// tensors themselves: a decode step's call 10.5 -> 5.0 us, the three calls of a chunk's ring work
// 22.0 -> 12.3 us, its kernels' time.  The checks are those of the Python code and of ctypes that
// they replace: a tensor that is not on the GPU raises ValueError, another structure than the
// descriptor's or a count that is no integer TypeError, a nonzero status PadraError.
#include <dlfcn.h>

#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <exception>
#include <tuple>
#include <type_traits>
#include <utility>

#include "padra_hip.h"

namespace {

struct PythonError {}; // the interpreter's error indicator is set

PyObject *g_error = nullptr; // abi.PadraError
// The descriptors' ctypes structures, as abi.py declares them.
template <class S> PyObject *g_structure = nullptr;

const at::Tensor *tensor(PyObject *o) {
  return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr;
}
[[noreturn]] void not_on_gpu() {
  PyErr_SetString(PyExc_ValueError, "padra_amd ops take GPU tensors");
  throw PythonError{};
}

// A tensor subclass or anything else with a tensor's attributes: through those.
void *address_by_attribute(PyObject *o) {
  PyObject *cuda = PyObject_GetAttrString(o, "is_cuda");
  if (!cuda)
    throw PythonError{};
  const int on = PyObject_IsTrue(cuda);
  Py_DECREF(cuda);
  if (on < 0)
    throw PythonError{};
  if (!on)
    not_on_gpu();
  PyObject *p = PyObject_CallMethod(o, "data_ptr", nullptr);
  if (!p)
    throw PythonError{};
  void *address = PyLong_AsVoidPtr(p);
  Py_DECREF(p);
  if (!address && PyErr_Occurred())
    throw PythonError{};
  return address;
}

void *address(PyObject *o) {
  if (o == Py_None)
    return nullptr;
  if (const at::Tensor *t = tensor(o)) {
    if (!t->is_cuda())
      not_on_gpu();
    return t->data_ptr();
  }
  return address_by_attribute(o);
}

// The current stream of the tensor's device.
void *stream_of(PyObject *o) {
  c10::DeviceIndex index = -1;
  if (const at::Tensor *t = tensor(o)) {
    if (!t->is_cuda())
      not_on_gpu();
    index = t->device().index();
  } else {
    address_by_attribute(o);
    PyObject *d = PyObject_CallMethod(o, "get_device", nullptr);
    if (!d)
      throw PythonError{};
    index = (c10::DeviceIndex)PyLong_AsLong(d);
    Py_DECREF(d);
    if (PyErr_Occurred())
      throw PythonError{};
  }
  return c10::hip::getCurrentHIPStream(index).stream();
}

// A descriptor: its own ctypes structure (or a subclass) and nothing else.  A KVCache is large
// enough for a Positions, and its plane pointers would be read as control records.
template <class S> const S *descriptor(PyObject *o) {
  if (o == Py_None)
    return nullptr;
  PyTypeObject *type = reinterpret_cast<PyTypeObject *>(g_structure<S>);
  if (!PyObject_TypeCheck(o, type)) {
    PyErr_Format(PyExc_TypeError, "expected %s, not %s", type->tp_name, Py_TYPE(o)->tp_name);
    throw PythonError{};
  }
  Py_buffer view;
  if (PyObject_GetBuffer(o, &view, PyBUF_SIMPLE) != 0)
    throw PythonError{};
  const S *s = static_cast<const S *>(view.buf);
  PyBuffer_Release(&view); // the structure's memory lives as long as the caller's object
  return s;
}

template <class A> A argument(PyObject *o) {
  if constexpr (std::is_same_v<A, const padra_Positions *>) {
    return descriptor<padra_Positions>(o);
  } else if constexpr (std::is_same_v<A, const padra_KVCache *>) {
    return descriptor<padra_KVCache>(o);
  } else if constexpr (std::is_pointer_v<A>) {
    return static_cast<A>(address(o));
  } else if constexpr (std::is_floating_point_v<A>) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1. && PyErr_Occurred())
      throw PythonError{};
    return (A)v;
  } else {
    PyObject *i = PyNumber_Index(o); // an integer, as ctypes asks: 1.9 or "2" is a TypeError
    if (!i)
      throw PythonError{};
    const unsigned long long v = PyLong_AsUnsignedLongLongMask(i);
    Py_DECREF(i);
    if (v == ~0ull && PyErr_Occurred())
      throw PythonError{};
    return (A)v;
  }
}

// One library function, bound at run time in the build that abi.library_path names.
template <auto Declared> struct Entry;
template <class R, class... A, R (*Declared)(A...)> struct Entry<Declared> {
  static inline R (*function)(A...) = nullptr;
  static inline const char *name = nullptr;

  // (Every argument is checked, left to right, before torch is asked for the stream.)
  template <bool LAUNCH, size_t... I>
  static R run(PyObject *const *args, std::index_sequence<I...>) {
    std::tuple<A...> values{LAUNCH && I == 0 ? A{} : argument<A>(args[I])...};
    if constexpr (LAUNCH)
      std::get<0>(values) = stream_of(args[0]);
    PyThreadState *state = PyEval_SaveThread(); // as ctypes does: a launch may wait for room
    const R r = function(std::get<I>(values)...);
    PyEval_RestoreThread(state);
    return r;
  }
  template <bool LAUNCH>
  static PyObject *call(PyObject *, PyObject *const *args, Py_ssize_t count) noexcept {
    if (!function || count != (Py_ssize_t)sizeof...(A)) {
      PyErr_Format(PyExc_TypeError, "%s takes %zd arguments (%zd given)", name ? name : "unbound",
                   (Py_ssize_t)sizeof...(A), count);
      return nullptr;
    }
    try {
      const R r = run<LAUNCH>(args, std::index_sequence_for<A...>{});
      if constexpr (!LAUNCH)
        return PyLong_FromLongLong(r);
      if (r != PADRA_OK) {
        PyObject *e = PyObject_CallFunction(g_error, "si", name, (int)r);
        if (e) {
          PyErr_SetObject(g_error, e);
          Py_DECREF(e);
        }
        return nullptr;
      }
      Py_RETURN_NONE;
    } catch (const PythonError &) {
    } catch (const std::exception &e) { // from a tensor without storage, for instance
      PyErr_SetString(PyExc_RuntimeError, e.what());
    }
    return nullptr;
  }
};

struct Listed {
  const char *name;
  void (*bind)(void *symbol, const char *name);
  PyMethodDef method;
};
template <auto Declared, bool LAUNCH> Listed listed(const char *name) {
  using E = Entry<Declared>;
  return {name,
          [](void *symbol, const char *n) {
            E::function = reinterpret_cast<decltype(E::function)>(symbol);
            E::name = n;
          },
          {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(&E::template call<LAUNCH>)),
           METH_FASTCALL, nullptr}};
}
#define LAUNCHED(fn) listed<&fn, true>(#fn)
#define VALUE(fn) listed<&fn, false>(#fn)

Listed g_listed[] = {
    LAUNCHED(padra_ResidualPostNorm),
    LAUNCHED(padra_NormFP8),
    LAUNCHED(padra_QuantizeFP8),
    LAUNCHED(padra_Combine),
    LAUNCHED(padra_CombineNorm),
    LAUNCHED(padra_QKNormRopeStore),
    LAUNCHED(padra_ResidualNormQKRopeStore),
    LAUNCHED(padra_EmbedResidualNormQKRopeStore),
    LAUNCHED(padra_KVStore),
    LAUNCHED(padra_KVCommit),
    LAUNCHED(padra_KVCheckpointCapture),
    LAUNCHED(padra_KvQ8_0Dequantize),
    LAUNCHED(padra_KvQ8_0DequantizePrefix),
    LAUNCHED(padra_DecodeAttention),
    LAUNCHED(padra_DecodeAttentionFP8),
    LAUNCHED(padra_RotateRows),
    LAUNCHED(padra_SiluTableBuild),
    LAUNCHED(padra_SwiGLU),
    LAUNCHED(padra_Embed),
    VALUE(padra_DecodeAttentionSplits),
    VALUE(padra_DecodeAttentionScratch),
};

// Whether o is a ctypes structure type of S's size.
template <class S> bool is_structure(PyObject *o) {
  PyObject *e = PyType_Check(o) ? PyObject_CallNoArgs(o) : nullptr;
  Py_buffer view;
  const bool same = e && PyObject_GetBuffer(e, &view, PyBUF_SIMPLE) == 0;
  const bool whole = same && view.len == (Py_ssize_t)sizeof(S);
  if (same)
    PyBuffer_Release(&view);
  Py_XDECREF(e);
  if (!whole && !PyErr_Occurred())
    PyErr_SetString(PyExc_TypeError, "bind takes the descriptors' ctypes structures");
  return whole;
}

// bind(library path, PadraError, Positions, KVCache) -> {entry point: function}
PyObject *bind(PyObject *, PyObject *args) {
  const char *path;
  PyObject *error, *positions, *cache;
  if (!PyArg_ParseTuple(args, "sOOO", &path, &error, &positions, &cache) ||
      !is_structure<padra_Positions>(positions) || !is_structure<padra_KVCache>(cache))
    return nullptr;
  void *library = dlopen(path, RTLD_NOW | RTLD_LOCAL);
  if (!library) {
    PyErr_SetString(PyExc_RuntimeError, dlerror());
    return nullptr;
  }
  PyObject *all = PyDict_New();
  for (Listed &l : g_listed) {
    void *symbol = dlsym(library, l.name);
    PyObject *f = symbol ? PyCFunction_New(&l.method, nullptr) : nullptr;
    if (!all || !f || PyDict_SetItemString(all, l.name, f) != 0) {
      if (!PyErr_Occurred())
        PyErr_Format(PyExc_RuntimeError, "%s has no %s", path, l.name);
      Py_XDECREF(f);
      Py_XDECREF(all);
      return nullptr;
    }
    Py_DECREF(f);
    l.bind(symbol, l.name);
  }
  Py_INCREF(error);
  Py_XSETREF(g_error, error);
  Py_INCREF(positions);
  Py_XSETREF(g_structure<padra_Positions>, positions);
  Py_INCREF(cache);
  Py_XSETREF(g_structure<padra_KVCache>, cache);
  return all;
}

PyMethodDef g_methods[] = {{"bind", bind, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_fastcall", nullptr, -1, g_methods,
                        nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__fastcall() { return PyModule_Create(&g_module); }
