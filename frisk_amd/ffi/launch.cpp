// The launches of frisk_amd/runtime.py as a CPython module: the same C ABI calls that ctypes makes, without its conversion of every argument through a type object.  A small
// call is bound by the host: of the 4.3 us that issuing a 128x128x128 product takes, the HIP launch is 3.
//
// Each function takes the arguments of its wrapper in runtime.py in their order and returns the library's status, or None for what it does not take -- another descriptor
// class, pointers that are no integers, more operands than a body can have -- which the wrapper then hands to ctypes as before.  Integers wrap as ctypes wraps
// them, and the interpreter lock is released during the call as ctypes releases it.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stdint.h>

#include "frisk_hip.h"

namespace {

// set by bind()
struct Library {
  decltype(&frisk_hip_gemm) gemm;
  decltype(&frisk_hip_fill) fill;
  decltype(&frisk_hip_copy) copy;
  decltype(&frisk_hip_reduce) reduce;
  decltype(&frisk_hip_elementwise) elementwise;
  decltype(&frisk_hip_softmax) softmax;
  decltype(&frisk_hip_attention) attention;
} lib;
PyTypeObject *gemm_desc, *elementwise_desc, *attention_desc;

// Arguments one after the other; `ok` turns false at the first that is not what ctypes would convert without asking its type
struct Args {
  PyObject* const* at;
  bool ok;
  Args(PyObject* const* args, Py_ssize_t n, Py_ssize_t want) : at(args), ok(n == want) {}
  void* pointer() {
    if (!ok) return nullptr;
    PyObject* o = *at++;
    if (o == Py_None) return nullptr;
    ok = PyLong_Check(o);
    return ok ? (void*)(uintptr_t)PyLong_AsUnsignedLongLongMask(o) : nullptr;
  }
  int64_t integer() {
    if (!ok) return 0;
    PyObject* o = *at++;
    ok = PyLong_Check(o);
    return ok ? (int64_t)PyLong_AsUnsignedLongLongMask(o) : 0;
  }
  double real() {
    if (!ok) return 0.0;
    PyObject* o = *at++;
    ok = PyFloat_Check(o);
    return ok ? PyFloat_AS_DOUBLE(o) : 0.0;
  }
};

// the memory of a ctypes structure, held while the call reads it
struct Struct {
  Py_buffer view{};
  bool held = false;
  Struct(Args& a, PyTypeObject* type, size_t size) {
    if (!a.ok) return;
    PyObject* o = *a.at++;
    held = Py_TYPE(o) == type && PyObject_GetBuffer(o, &view, PyBUF_SIMPLE) == 0;
    if (PyErr_Occurred()) PyErr_Clear();
    a.ok = held && (size_t)view.len == size;
  }
  ~Struct() { if (held) PyBuffer_Release(&view); }
};

template <class F> PyObject* call(const Args& a, F&& f) {
  if (!a.ok || !lib.gemm) Py_RETURN_NONE;
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = f();
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(status);
}

PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Args a(args, n, 9);
  const Struct d(a, gemm_desc, sizeof(frisk_gemm_desc));
  void *A = a.pointer(), *B = a.pointer(), *C = a.pointer(), *sa = a.pointer(), *sb = a.pointer(), *ws = a.pointer();
  const size_t ws_bytes = (size_t)a.integer();
  void* stream = a.pointer();
  return call(a, [&] { return lib.gemm((const frisk_gemm_desc*)d.view.buf, A, B, C, (const float*)sa, (const float*)sb, ws, ws_bytes, stream); });
}

PyObject* fill(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Args a(args, n, 7);
  const int dtype = (int)a.integer();
  void* dst = a.pointer();
  const int64_t rows = a.integer(), cols = a.integer(), ld = a.integer();
  const double value = a.real();
  void* stream = a.pointer();
  return call(a, [&] { return lib.fill(dtype, dst, rows, cols, ld, value, stream); });
}

PyObject* copy(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Args a(args, n, 9);
  const int sdt = (int)a.integer();
  void* src = a.pointer();
  const int64_t sld = a.integer();
  const int ddt = (int)a.integer();
  void* dst = a.pointer();
  const int64_t dld = a.integer(), rows = a.integer(), cols = a.integer();
  void* stream = a.pointer();
  return call(a, [&] { return lib.copy(sdt, src, sld, ddt, dst, dld, rows, cols, stream); });
}

PyObject* reduce(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Args a(args, n, 12);
  const int dtype = (int)a.integer();
  void* src = a.pointer();
  const int64_t rows = a.integer(), cols = a.integer(), ld = a.integer();
  const int dim = (int)a.integer(), kind = (int)a.integer(), clear = (int)a.integer();
  void *dst = a.pointer(), *ws = a.pointer();
  const size_t ws_bytes = (size_t)a.integer();
  void* stream = a.pointer();
  return call(a, [&] { return lib.reduce(dtype, src, rows, cols, ld, dim, kind, clear, dst, ws, ws_bytes, stream); });
}

PyObject* elementwise(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Args a(args, n, 4);
  const Struct d(a, elementwise_desc, sizeof(frisk_elementwise_desc));
  const void* in[FRISK_EW_MAX_INPUTS] = {};
  if (a.ok) {
    PyObject* o = *a.at++;
    const bool list = PyList_CheckExact(o);
    const Py_ssize_t count = list ? PyList_GET_SIZE(o) : PyTuple_CheckExact(o) ? PyTuple_GET_SIZE(o) : -1;
    a.ok = count >= 0 && count <= FRISK_EW_MAX_INPUTS;
    if (a.ok) {
      Args each(list ? ((PyListObject*)o)->ob_item : ((PyTupleObject*)o)->ob_item, count, count);
      for (Py_ssize_t i = 0; i < count; ++i) in[i] = each.pointer();
      a.ok = each.ok;
    }
  }
  void *out = a.pointer(), *stream = a.pointer();
  return call(a, [&] { return lib.elementwise((const frisk_elementwise_desc*)d.view.buf, in, out, stream); });
}

PyObject* softmax(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Args a(args, n, 12);
  const int dtype = (int)a.integer();
  void* src = a.pointer();
  const int64_t sld = a.integer();
  void* dst = a.pointer();
  const int64_t dld = a.integer(), rows = a.integer(), cols = a.integer();
  const float scale = (float)a.real();
  void *lse = a.pointer(), *ws = a.pointer();
  const size_t ws_bytes = (size_t)a.integer();
  void* stream = a.pointer();
  return call(a, [&] { return lib.softmax(dtype, src, sld, dst, dld, rows, cols, scale, (float*)lse, ws, ws_bytes, stream); });
}

PyObject* attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Args a(args, n, 7);
  const Struct d(a, attention_desc, sizeof(frisk_attention_desc));
  void *q = a.pointer(), *k = a.pointer(), *v = a.pointer(), *o = a.pointer(), *lse = a.pointer(), *stream = a.pointer();
  return call(a, [&] { return lib.attention((const frisk_attention_desc*)d.view.buf, q, k, v, o, (float*)lse, stream); });
}

// bind(GemmDesc, ElementwiseDesc, AttentionDesc, addresses of gemm, fill, copy, reduce, elementwise, softmax, attention)
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 10 || !PyType_Check(args[0]) || !PyType_Check(args[1]) || !PyType_Check(args[2])) {
    PyErr_SetString(PyExc_TypeError, "bind takes three descriptor classes and seven addresses");
    return nullptr;
  }
  Args a(args + 3, n - 3, 7);
  void* f[7];
  for (void*& p : f) p = a.pointer();
  if (!a.ok) {
    PyErr_SetString(PyExc_TypeError, "bind takes three descriptor classes and seven addresses");
    return nullptr;
  }
  PyTypeObject** const types[3] = {&gemm_desc, &elementwise_desc, &attention_desc};
  for (int i = 0; i < 3; ++i) {
    Py_INCREF(args[i]);
    Py_XDECREF(*types[i]);
    *types[i] = (PyTypeObject*)args[i];
  }
  lib = Library{(decltype(lib.gemm))f[0], (decltype(lib.fill))f[1], (decltype(lib.copy))f[2], (decltype(lib.reduce))f[3], (decltype(lib.elementwise))f[4],
                (decltype(lib.softmax))f[5], (decltype(lib.attention))f[6]};
  Py_RETURN_NONE;
}

#define FRISK_FUNCTION(NAME) {#NAME, (PyCFunction)(void (*)(void))NAME, METH_FASTCALL, nullptr}
PyMethodDef functions[] = {FRISK_FUNCTION(bind), FRISK_FUNCTION(gemm), FRISK_FUNCTION(fill), FRISK_FUNCTION(copy), FRISK_FUNCTION(reduce), FRISK_FUNCTION(elementwise),
                           FRISK_FUNCTION(softmax), FRISK_FUNCTION(attention), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "frisk_launch", "launches of libfrisk_hip.so for frisk_amd.runtime", -1, functions, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_frisk_launch(void) { return PyModule_Create(&module); }
