// The method a module is called most often by, from numpy arrays to the py_ function and back.
//
// Coercing six arguments and describing them as memrefs in Python and ctypes takes 60 us; a product of a small matrix on
// host arrays takes about as long.  Here the arrays are read through the buffer protocol.  Arguments that need coercing
// (lists, other element types, other layouts) are left to the caller.
#include <Python.h>

#include <cstring>

#include "lapis_module.h"

namespace {

struct Buffer {
  Py_buffer view{};
  bool held = false;
  ~Buffer() {
    if (held) PyBuffer_Release(&view);
  }
  // a one-dimensional C-contiguous array of `format`?
  bool take(PyObject *o, bool writable) {
    if (!PyObject_CheckBuffer(o)) return false;
    if (PyObject_GetBuffer(o, &view, PyBUF_C_CONTIGUOUS | PyBUF_FORMAT | (writable ? PyBUF_WRITABLE : 0)) != 0) {
      PyErr_Clear();
      return false;
    }
    held = true;
    return view.ndim == 1;
  }
  bool holds(char format, Py_ssize_t size) const {
    return view.itemsize == size && view.format && view.format[0] == format && view.format[1] == 0;
  }
  template <typename M>
  M memref() const {
    M m;
    m.basePtr = m.data = static_cast<decltype(m.data)>(view.buf);
    m.offset = 0;
    m.sizes[0] = view.shape[0];
    m.strides[0] = 1;
    return m;
  }
};

bool integers(PyObject *sequence, Py_ssize_t count, int64_t *out) {
  PyObject *fast = PySequence_Fast(sequence, "a storage specifier");
  if (!fast) return false;
  bool ok = PySequence_Fast_GET_SIZE(fast) >= count;
  for (Py_ssize_t i = 0; ok && i < count; ++i) {
    PyObject *index = PyNumber_Index(PySequence_Fast_GET_ITEM(fast, i));
    out[i] = index ? PyLong_AsLongLong(index) : -1;
    Py_XDECREF(index);
    ok = !PyErr_Occurred();
  }
  Py_DECREF(fast);
  return ok;
}

bool specifier(PyObject *o, lapis_csr_specifier *spec) {
  if (!PyTuple_Check(o) || PyTuple_GET_SIZE(o) < 2) return false;
  int64_t flat[5];
  if (!integers(PyTuple_GET_ITEM(o, 0), 2, flat) || !integers(PyTuple_GET_ITEM(o, 1), 3, flat + 2)) {
    PyErr_Clear();
    return false;
  }
  static_assert(sizeof(lapis_csr_specifier) == sizeof(flat), "five 64-bit words");
  memcpy(spec, flat, sizeof(flat));
  return true;
}

template <typename M>
void call(void *entry, const Buffer &pos, const Buffer &crd, const Buffer &val, const lapis_csr_specifier *spec,
          const Buffer &x, const Buffer &y) {
  typedef void (*Entry)(M **, lapis_memref_1d_i32 *, lapis_memref_1d_i32 *, M *, const lapis_csr_specifier *, M *, M *);
  auto p = pos.memref<lapis_memref_1d_i32>(), c = crd.memref<lapis_memref_1d_i32>();
  M v = val.memref<M>(), xm = x.memref<M>(), ym = y.memref<M>(), out{}, *ret = &out;
  Py_BEGIN_ALLOW_THREADS;
  reinterpret_cast<Entry>(entry)(&ret, &p, &c, &v, spec, &xm, &ym);
  Py_END_ALLOW_THREADS;
}

// spmv(py_spmv, py_spmv_f32, positions, coordinates, values, specifier, x, y) -> True, or False if nothing was done
PyObject *py_spmv(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (n != 8) {
    PyErr_SetString(PyExc_TypeError, "spmv: 8 arguments");
    return nullptr;
  }
  void *f64 = PyLong_AsVoidPtr(a[0]), *f32 = PyLong_AsVoidPtr(a[1]);
  if (PyErr_Occurred()) return nullptr;
  Buffer pos, crd, val, x, y;
  lapis_csr_specifier spec;
  if (!pos.take(a[2], false) || !crd.take(a[3], false) || !val.take(a[4], false) || !x.take(a[6], false) ||
      !y.take(a[7], true) || !specifier(a[5], &spec) || !pos.holds('i', 4) || !crd.holds('i', 4))
    Py_RETURN_FALSE;
  if (val.holds('d', 8) && x.holds('d', 8) && y.holds('d', 8))
    call<lapis_memref_1d_f64>(f64, pos, crd, val, &spec, x, y);
  else if (val.holds('f', 4) && x.holds('f', 4) && y.holds('f', 4))
    call<lapis_memref_1d_f32>(f32, pos, crd, val, &spec, x, y);
  else
    Py_RETURN_FALSE;
  Py_RETURN_TRUE;
}

PyMethodDef g_methods[] = {{"spmv", (PyCFunction)(void (*)(void))py_spmv, METH_FASTCALL, nullptr},
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_lapis_module_calls", "Calls of module functions on numpy arrays.", -1,
                        g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__lapis_module_calls(void) { return PyModule_Create(&g_module); }
