// host.cpp -- the module's launch path as a CPython extension: every ldr_* entry point as a builtin that takes tensors,
// None, numbers and address tables as they are, and the allocations around a read. A launch through ctypes costs 4-5 us
// of argument conversion (up to 30 arguments, each tensor's address fetched in Python before), and a small pass is a few
// dozen of them: these cost about 1 us.
//
// The entry points' addresses come from the library the Python binding loaded (bind), so both always call the same one.

#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>

#include <cstring>
#include <tuple>
#include <utility>

#include "loopback_read.h"

namespace {

// one argument of an entry point, converted from a Python object; set() leaves a Python error on failure
template <typename A> struct Arg;

template <typename P> struct Arg<P*> {   // a device address: a tensor's, an int, or None
  P* v = nullptr;
  bool set(PyObject* o) {
    if (o == Py_None) return true;
    if (THPVariable_Check(o)) {
      v = static_cast<P*>(THPVariable_Unpack(o).data_ptr());
      return true;
    }
    v = static_cast<P*>(PyLong_AsVoidPtr(o));
    return !(v == nullptr && PyErr_Occurred());
  }
};

// A table of addresses: a list or tuple of tensors and ints (at most LDR_MAX_SOURCES), an array of 64-bit integers
// (anything with a buffer, as the stack's cached tables), or a device array's address as an int.
template <> struct Arg<const uint64_t*> {
  const uint64_t* v = nullptr;
  uint64_t own[LDR_MAX_SOURCES];
  Py_buffer buf{};
  bool held = false;
  ~Arg() { if (held) PyBuffer_Release(&buf); }
  bool set(PyObject* o) {
    if (o == Py_None) return true;
    const bool list = PyList_CheckExact(o);
    if (list || PyTuple_CheckExact(o)) {
      const Py_ssize_t n = list ? PyList_GET_SIZE(o) : PyTuple_GET_SIZE(o);
      if (n > LDR_MAX_SOURCES) {
        PyErr_SetString(PyExc_ValueError, "an address table of more than LDR_MAX_SOURCES entries");
        return false;
      }
      for (Py_ssize_t i = 0; i < n; ++i) {
        Arg<void*> e;
        if (!e.set(list ? PyList_GET_ITEM(o, i) : PyTuple_GET_ITEM(o, i))) return false;
        own[i] = reinterpret_cast<uint64_t>(e.v);
      }
      v = own;
      return true;
    }
    if (PyLong_Check(o)) {
      v = static_cast<const uint64_t*>(PyLong_AsVoidPtr(o));
      return !(v == nullptr && PyErr_Occurred());
    }
    if (PyObject_GetBuffer(o, &buf, PyBUF_SIMPLE) != 0) return false;
    held = true;
    v = static_cast<const uint64_t*>(buf.buf);
    return true;
  }
};

template <> struct Arg<int64_t> {
  int64_t v = 0;
  bool set(PyObject* o) {
    v = PyLong_AsLongLong(o);
    return !(v == -1 && PyErr_Occurred());
  }
};
template <> struct Arg<int> {
  int v = 0;
  bool set(PyObject* o) {
    const long x = PyLong_AsLong(o);
    if (x == -1 && PyErr_Occurred()) return false;
    v = static_cast<int>(x);
    return true;
  }
};
template <> struct Arg<float> {
  float v = 0.f;
  bool set(PyObject* o) {
    const double x = PyFloat_AsDouble(o);
    if (x == -1.0 && PyErr_Occurred()) return false;
    v = static_cast<float>(x);
    return true;
  }
};

template <typename... A, size_t... I>
PyObject* invoke(int (*f)(A...), PyObject* const* args, std::index_sequence<I...>) {
  std::tuple<Arg<A>...> t;
  if (!(std::get<I>(t).set(args[I]) && ...)) return nullptr;
  int code;
  Py_BEGIN_ALLOW_THREADS
  code = f(std::get<I>(t).v...);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(code);
}

// one entry point: its address once bound, and the builtin that calls it
template <typename F, int ID> struct Entry;
template <typename... A, int ID> struct Entry<int (*)(A...), ID> {
  static inline int (*fn)(A...) = nullptr;
  static PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (!fn || n != static_cast<Py_ssize_t>(sizeof...(A))) {
      PyErr_Format(PyExc_TypeError, fn ? "entry point takes %zd arguments, got %zd" : "entry point not bound",
                   static_cast<Py_ssize_t>(sizeof...(A)), n);
      return nullptr;
    }
    return invoke(fn, args, std::index_sequence_for<A...>());
    END_HANDLE_TH_ERRORS
  }
  static void bind(void* p) { fn = reinterpret_cast<int (*)(A...)>(p); }
};

#define LDR_ENTRIES(X)                                                                                           \
  X(rstd_fwd) X(rstd_bwd) X(write_dots) X(split_queries) X(dots_online) X(read_fwd) X(read_fwd_online)             \
  X(read_bwd1) X(read_bwd1_noalloc) X(reduce_rows) X(blend_sum) X(read_bwd2_list) X(dv_assemble) X(read_fwd_any)   \
  X(read_bwd1_any) X(dv_assemble_any) X(read_bwd2_list_any) X(blend_sum_any) X(write_rows) X(read_fwd_rows)        \
  X(read_bwd1_rows) X(dv_assemble_rows) X(read_bwd2_list_rows) X(blend_sum_rows)

enum Id {
#define X(name) ID_##name,
  LDR_ENTRIES(X)
#undef X
};

struct Binding { const char* name; void (*bind)(void*); };
const Binding bindings[] = {
#define X(name) {"ldr_" #name, &Entry<decltype(&ldr_##name), ID_##name>::bind},
    LDR_ENTRIES(X)
#undef X
};

// bind(name, address) of an entry point; False for a name this module has no builtin for
PyObject* host_bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 2) {
    PyErr_SetString(PyExc_TypeError, "bind(name, address)");
    return nullptr;
  }
  const char* name = PyUnicode_AsUTF8(args[0]);
  if (!name) return nullptr;
  void* p = PyLong_AsVoidPtr(args[1]);
  if (!p && PyErr_Occurred()) return nullptr;
  for (const Binding& b : bindings)
    if (std::strcmp(b.name, name) == 0) {
      b.bind(p);
      Py_RETURN_TRUE;
    }
  Py_RETURN_FALSE;
}

// alias(t, s): t[s] as a tensor of its own on t's storage (no autograd view of t, its own version counter)
PyObject* host_alias(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !THPVariable_Check(args[0])) {
    PyErr_SetString(PyExc_TypeError, "alias(tensor, index)");
    return nullptr;
  }
  const at::Tensor& t = THPVariable_Unpack(args[0]);
  int64_t s = PyLong_AsLongLong(args[1]);
  if (s == -1 && PyErr_Occurred()) return nullptr;
  if (s < 0 && t.dim() > 0) s += t.size(0);
  if (t.dim() < 1 || s < 0 || s >= t.size(0)) {
    PyErr_SetString(PyExc_IndexError, "alias: index out of range");
    return nullptr;
  }
  at::Tensor out = at::empty({0}, t.options());
  out.set_(t.storage(), t.storage_offset() + s * t.stride(0), t.sizes().slice(1), t.strides().slice(1));
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// read_buffers(like, n_tok, n, prob, prior, dots): a read's outputs (out, tc, prob or None, next prior or None, raw
// scores or None)
PyObject* host_read_buffers(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6 || !THPVariable_Check(args[0])) {
    PyErr_SetString(PyExc_TypeError, "read_buffers(like, n_tok, n, prob, prior, dots)");
    return nullptr;
  }
  const at::Tensor& like = THPVariable_Unpack(args[0]);
  const int64_t n_tok = PyLong_AsLongLong(args[1]), ns = PyLong_AsLongLong(args[2]);
  if (PyErr_Occurred()) return nullptr;
  const auto f32 = at::TensorOptions().dtype(at::kFloat).device(like.device());
  PyObject* out = PyTuple_New(5);
  if (!out) return nullptr;
  try {
    PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(at::empty_like(like)));
    PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(at::empty({n_tok, ns}, f32)));
    auto opt = [&](int i, PyObject* flag, at::IntArrayRef shape) {
      PyObject* o = Py_None;
      if (flag == Py_True) o = THPVariable_Wrap(at::empty(shape, f32));
      else Py_INCREF(o);
      PyTuple_SET_ITEM(out, i, o);
    };
    opt(2, args[3], {n_tok, ns});
    opt(3, args[4], {ns});
    opt(4, args[5], {ns, n_tok});
  } catch (...) {
    Py_DECREF(out);
    throw;
  }
  return out;
  END_HANDLE_TH_ERRORS
}

#define FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f))
PyMethodDef methods[] = {
#define X(name) {#name, FAST((&Entry<decltype(&ldr_##name), ID_##name>::call)), METH_FASTCALL, nullptr},
    LDR_ENTRIES(X)
#undef X
    {"bind", FAST(&host_bind), METH_FASTCALL, nullptr},
    {"alias", FAST(&host_alias), METH_FASTCALL, nullptr},
    {"read_buffers", FAST(&host_read_buffers), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "launch path of the Loopback read", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }
