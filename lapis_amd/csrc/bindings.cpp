// Python entry points of the device-resident calls, on the CPython and PyTorch C++ APIs.
//
// A call of a small matrix takes the GPU 4 us; checking its operands, looking up the stream and converting nine
// arguments in Python and ctypes took 9 us.  The functions here do the same checks on the tensors themselves, take
// torch's current stream and call the C ABI directly (include/lapis_hip.h).  lapis_amd/hip.py wraps them and
// documents them; operands that are plain integers pass as raw device addresses, as they do there.
#include <Python.h>

#include <ATen/ops/empty.h>
#include <ATen/ops/from_blob.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdarg>
#include <memory>
#include <vector>

#include "blas1.hpp"
#include "lapis_hip.h"
#include "staging.hpp"

namespace {

PyObject *g_check = nullptr;  // lapis_amd.hip.check: raises LapisHipError for a status that is not OK
PyObject *g_init = nullptr;   // lapis_amd.hip.init, called before the first call that reaches the device
bool g_ready = false;

// thrown once a Python error is set
struct Raised {};

[[noreturn]] void raise(PyObject *type, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  PyErr_FormatV(type, fmt, ap);
  va_end(ap);
  throw Raised();
}

// An operand: a tensor, a raw address or None.
struct Operand {
  const at::Tensor *tensor = nullptr;
  void *address = nullptr;
};

Operand operand(PyObject *o) {
  Operand r;
  if (o == Py_None) return r;
  if (THPVariable_Check(o)) {
    r.tensor = &THPVariable_Unpack(o);
    r.address = r.tensor->data_ptr();
    return r;
  }
  if (PyLong_Check(o)) {
    r.address = PyLong_AsVoidPtr(o);
    if (PyErr_Occurred()) throw Raised();
    return r;
  }
  raise(PyExc_TypeError, "an operand is neither a tensor, a device address nor None but %s", Py_TYPE(o)->tp_name);
}

int64_t integer(PyObject *o) {
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) {
    // numpy integers and the like
    PyErr_Clear();
    PyObject *i = PyNumber_Index(o);
    if (!i) throw Raised();
    const long long w = PyLong_AsLongLong(i);
    Py_DECREF(i);
    if (w == -1 && PyErr_Occurred()) throw Raised();
    return w;
  }
  return v;
}

double number(PyObject *o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw Raised();
  return v;
}

// Every call asks for its stream after its operands have passed their checks: malformed operands are refused
// without a GPU too.
lapis_hip_stream_t stream_of(PyObject *o) {
  if (!g_ready) {
    PyObject *r = PyObject_CallNoArgs(g_init);
    if (!r) throw Raised();
    Py_DECREF(r);
    g_ready = true;
  }
  if (o == Py_None) return c10::hip::getCurrentHIPStream().stream();
  if (PyLong_Check(o)) return PyLong_AsVoidPtr(o);
  PyObject *raw = PyObject_GetAttrString(o, "cuda_stream");  // a torch.cuda.Stream
  if (!raw) throw Raised();
  void *p = PyLong_AsVoidPtr(raw);
  Py_DECREF(raw);
  if (PyErr_Occurred()) throw Raised();
  return p;
}

lapis_hip_csr_plan *plan_of(PyObject *o) {
  if (o == Py_None) return nullptr;
  static PyObject *name = PyUnicode_InternFromString("address");
  PyObject *a = PyObject_GetAttr(o, name);
  if (!a) throw Raised();
  void *p = a == Py_None ? nullptr : PyLong_AsVoidPtr(a);
  Py_DECREF(a);
  if (PyErr_Occurred()) throw Raised();
  return static_cast<lapis_hip_csr_plan *>(p);
}

const char *type_name(at::ScalarType t) { return c10::toString(t); }

// The C ABI takes pointers and counts: a tensor with fewer than `n` elements, of another element type than `like`
// or with gaps between its elements would be read or written past its end on the device.
void holds(const char *what, int64_t n, const Operand &o, const at::Tensor *like = nullptr) {
  if (!o.tensor) return;
  const at::Tensor &t = *o.tensor;
  if (t.numel() < n)
    raise(PyExc_ValueError, "%s: an operand of %lld elements where %lld are needed", what, (long long)t.numel(), (long long)n);
  if (like && t.scalar_type() != like->scalar_type())
    raise(PyExc_TypeError, "%s: operands of %s and %s", what, type_name(t.scalar_type()), type_name(like->scalar_type()));
  if (!t.is_contiguous()) raise(PyExc_ValueError, "%s: an operand that is not contiguous", what);
}

void indices(const char *what, const Operand &o) {
  if (o.tensor && o.tensor->scalar_type() != at::kInt)
    raise(PyExc_TypeError, "%s: positions and coordinates are int32, got %s", what, type_name(o.tensor->scalar_type()));
}

// fp32 or fp64 by the element type of `o`
bool is_f64(const Operand &o) {
  if (!o.tensor) raise(PyExc_TypeError, "values must be a float32 or float64 tensor");
  const auto t = o.tensor->scalar_type();
  if (t != at::kDouble && t != at::kFloat) raise(PyExc_TypeError, "values must be float32 or float64, got %s", type_name(t));
  return t == at::kDouble;
}

int64_t length(const char *what, const Operand &o) {
  if (!o.tensor || o.tensor->dim() < 1) raise(PyExc_TypeError, "%s: an operand that is not a tensor of at least one dimension", what);
  return o.tensor->size(0);
}

void check(int status) {
  if (status == LAPIS_HIP_OK) return;
  PyObject *r = PyObject_CallFunction(g_check, "i", status);
  Py_XDECREF(r);
  if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "lapis_hip call failed");
  throw Raised();
}

PyObject *give(PyObject *o) {
  Py_INCREF(o);
  return o;
}

void arguments(const char *what, Py_ssize_t got, Py_ssize_t want) {
  if (got != want) raise(PyExc_TypeError, "%s: %zd arguments, %zd expected", what, got, want);
}

template <typename F>
PyObject *guarded(F f) {
  try {
    return f();
  } catch (const Raised &) {
    return nullptr;
  } catch (const std::exception &e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

// A dot product under way is a capsule: one that nobody finishes is waited for when it goes.
constexpr const char *kSumName = "lapis_hip.dot";
void abandon_sum(PyObject *capsule) {
  lapis::dot_abandon(static_cast<lapis::HostSum *>(PyCapsule_GetPointer(capsule, kSumName)));
}
PyObject *sum_capsule(lapis::HostSum *sum) {
  PyObject *c = PyCapsule_New(sum, kSumName, abandon_sum);
  if (!c) {
    lapis::dot_abandon(sum);
    throw Raised();
  }
  return c;
}

#define LAPIS_PY(name) PyObject *name(PyObject *, PyObject *const *a, Py_ssize_t n)

struct SpmvCall {
  lapis_hip_csr_plan *plan;
  int64_t nrows, ncols;
  const int32_t *pos, *crd;
  Operand val, x, y;
  // a[0..7]: plan, nrows, ncols, pos, crd, val, x, y
  explicit SpmvCall(PyObject *const *a) {
    nrows = integer(a[1]);
    ncols = integer(a[2]);
    const Operand p = operand(a[3]), c = operand(a[4]);
    val = operand(a[5]);
    x = operand(a[6]);
    y = operand(a[7]);
    indices("spmv", p);
    indices("spmv", c);
    holds("spmv", nrows + 1, p);
    holds("spmv", ncols, x, val.tensor);
    holds("spmv", nrows, y, val.tensor);
    if (c.tensor) holds("spmv", c.tensor->numel(), val);
    plan = plan_of(a[0]);
    pos = static_cast<const int32_t *>(p.address);
    crd = static_cast<const int32_t *>(c.address);
  }
};

// (plan, nrows, ncols, pos, crd, val, x, y, stream)
LAPIS_PY(py_spmv) {
  return guarded([&] {
    arguments("spmv", n, 9);
    const SpmvCall c(a);
    if (is_f64(c.val))
      check(lapis_hip_spmv_csr_f64_i32(c.plan, c.nrows, c.ncols, c.pos, c.crd, (const double *)c.val.address,
                                       (const double *)c.x.address, (double *)c.y.address, stream_of(a[8])));
    else
      check(lapis_hip_spmv_csr_f32_i32(c.plan, c.nrows, c.ncols, c.pos, c.crd, (const float *)c.val.address,
                                       (const float *)c.x.address, (float *)c.y.address, stream_of(a[8])));
    return give(a[7]);
  });
}

// (plan, nrows, ncols, pos, crd, val, x, y, stream): y = A x
LAPIS_PY(py_spmv_overwrite) {
  return guarded([&] {
    arguments("spmv", n, 9);
    const SpmvCall c(a);
    if (is_f64(c.val))
      check(lapis::spmv_overwrite<double>(c.plan, c.nrows, c.ncols, c.pos, c.crd, (const double *)c.val.address,
                                          (const double *)c.x.address, (double *)c.y.address, stream_of(a[8])));
    else
      check(lapis::spmv_overwrite<float>(c.plan, c.nrows, c.ncols, c.pos, c.crd, (const float *)c.val.address,
                                         (const float *)c.x.address, (float *)c.y.address, stream_of(a[8])));
    return give(a[7]);
  });
}

// (plan, nrows, ncols, pos, crd, val, x, y, init, stream) -> capsule of init + x . y: y = A x
LAPIS_PY(py_spmv_dot_start) {
  return guarded([&] {
    arguments("spmv", n, 10);
    const SpmvCall c(a);
    const double init = number(a[8]);
    lapis::HostSum *sum = nullptr;
    if (is_f64(c.val))
      check(lapis::spmv_dot_start<double>(c.plan, c.nrows, c.ncols, c.pos, c.crd, (const double *)c.val.address,
                                          (const double *)c.x.address, (double *)c.y.address, init, stream_of(a[9]), &sum));
    else
      check(lapis::spmv_dot_start<float>(c.plan, c.nrows, c.ncols, c.pos, c.crd, (const float *)c.val.address,
                                         (const float *)c.x.address, (float *)c.y.address, init, stream_of(a[9]), &sum));
    return sum_capsule(sum);
  });
}

// (nrows, ncols, pos, crd, val, B, C, stream, plan)
LAPIS_PY(py_spmm) {
  return guarded([&] {
    arguments("spmm", n, 9);
    const int64_t nrows = integer(a[0]), ncols = integer(a[1]);
    const Operand pos = operand(a[2]), crd = operand(a[3]), val = operand(a[4]), B = operand(a[5]), C = operand(a[6]);
    if (!B.tensor || !C.tensor || !crd.tensor || !val.tensor) raise(PyExc_TypeError, "spmm: crd, val, B and C are tensors");
    indices("spmm", pos);
    indices("spmm", crd);
    holds("spmm", nrows + 1, pos);
    holds("spmm", crd.tensor->numel(), val);
    const at::Tensor &b = *B.tensor, &c = *C.tensor, &v = *val.tensor;
    if (b.dim() != 2 || c.dim() != 2 || b.size(1) != c.size(1) || b.size(0) < ncols || c.size(0) < nrows ||
        b.stride(1) != 1 || c.stride(1) != 1 || b.scalar_type() != v.scalar_type() || c.scalar_type() != v.scalar_type())
      raise(PyExc_ValueError, "spmm: a %lld x %lld matrix of %s times B (%d dimensions, %lld elements) into C (%d, %lld)",
            (long long)nrows, (long long)ncols, type_name(v.scalar_type()), (int)b.dim(), (long long)b.numel(), (int)c.dim(),
            (long long)c.numel());
    const int64_t k = c.size(1);
    lapis_hip_csr_plan *plan = plan_of(a[8]);
    const auto p = static_cast<const int32_t *>(pos.address), cr = static_cast<const int32_t *>(crd.address);
    if (is_f64(val))
      check(lapis_hip_spmm_csr_f64_i32_plan(plan, nrows, ncols, k, p, cr, (const double *)val.address, (const double *)B.address,
                                            b.stride(0), (double *)C.address, c.stride(0), stream_of(a[7])));
    else
      check(lapis_hip_spmm_csr_f32_i32_plan(plan, nrows, ncols, k, p, cr, (const float *)val.address, (const float *)B.address,
                                            b.stride(0), (float *)C.address, c.stride(0), stream_of(a[7])));
    return give(a[6]);
  });
}

// (n1, n2, pos, crd, val, V, out, stream)
LAPIS_PY(py_bspmm_csrv) {
  return guarded([&] {
    arguments("bspmm_csrv", n, 8);
    const int64_t n1 = integer(a[0]), n2 = integer(a[1]);
    const Operand pos = operand(a[2]), crd = operand(a[3]), val = operand(a[4]), V = operand(a[5]), out = operand(a[6]);
    if (!V.tensor || V.tensor->dim() != 3) raise(PyExc_IndexError, "bspmm_csrv: V has three dimensions");
    check(lapis_hip_bspmm_csrv_f32_i32(n1, n2, V.tensor->size(1), V.tensor->size(2), (const int32_t *)pos.address,
                                       (const int32_t *)crd.address, (const float *)val.address, (const float *)V.address,
                                       (float *)out.address, stream_of(a[7])));
    return give(a[6]);
  });
}

// (x, y, result, init, stream)
LAPIS_PY(py_dot) {
  return guarded([&] {
    arguments("dot", n, 5);
    const Operand x = operand(a[0]), y = operand(a[1]), r = operand(a[2]);
    const int64_t len = length("dot", x);
    holds("dot", len, x, x.tensor);
    holds("dot", len, y, x.tensor);
    holds("dot", 1, r, x.tensor);
    const double init = number(a[3]);
    if (is_f64(x))
      check(lapis_hip_dot_f64(len, (const double *)x.address, (const double *)y.address, init, (double *)r.address, stream_of(a[4])));
    else
      check(lapis_hip_dot_f32(len, (const float *)x.address, (const float *)y.address, (float)init, (float *)r.address,
                              stream_of(a[4])));
    return give(a[2]);
  });
}

// (x, y, init, stream) -> float.  The call waits for the GPU: other Python threads run meanwhile.
LAPIS_PY(py_dot_host) {
  return guarded([&] {
    arguments("dot", n, 4);
    const Operand x = operand(a[0]), y = operand(a[1]);
    const int64_t len = length("dot", x);
    holds("dot", len, x, x.tensor);
    holds("dot", len, y, x.tensor);
    const double init = number(a[2]);
    const lapis_hip_stream_t st = stream_of(a[3]);
    double r64 = 0.0;
    float r32 = 0.f;
    const bool f64 = is_f64(x);
    int status;
    Py_BEGIN_ALLOW_THREADS;
    status = f64 ? lapis_hip_dot_f64_host(len, (const double *)x.address, (const double *)y.address, init, &r64, st)
                 : lapis_hip_dot_f32_host(len, (const float *)x.address, (const float *)y.address, (float)init, &r32, st);
    Py_END_ALLOW_THREADS;
    check(status);
    return PyFloat_FromDouble(f64 ? r64 : (double)r32);
  });
}

// (x, y, init, stream) -> capsule of init + x . y
LAPIS_PY(py_dot_start) {
  return guarded([&] {
    arguments("dot", n, 4);
    const Operand x = operand(a[0]), y = operand(a[1]);
    const int64_t len = length("dot", x);
    holds("dot", len, x, x.tensor);
    holds("dot", len, y, x.tensor);
    const double init = number(a[2]);
    const hipStream_t st = static_cast<hipStream_t>(stream_of(a[3]));
    lapis::HostSum *sum = nullptr;
    check(is_f64(x) ? lapis::dot_start<double>(len, (const double *)x.address, (const double *)y.address, init, st, &sum)
                    : lapis::dot_start<float>(len, (const float *)x.address, (const float *)y.address, init, st, &sum));
    return sum_capsule(sum);
  });
}

// (a, x, b, y, dst, z or None, init, stream) -> capsule of init + dst . z (dst . dst without z): dst = a x + b y
LAPIS_PY(py_axpby_dot_start) {
  return guarded([&] {
    arguments("axpby_dot", n, 8);
    const double ca = number(a[0]), cb = number(a[2]);
    const Operand x = operand(a[1]), y = operand(a[3]), d = operand(a[4]), z = operand(a[5]);
    const int64_t len = length("axpby_dot", x);
    holds("axpby_dot", len, x, x.tensor);
    holds("axpby_dot", len, y, x.tensor);
    holds("axpby_dot", len, d, x.tensor);
    holds("axpby_dot", len, z, x.tensor);
    const double init = number(a[6]);
    const hipStream_t st = static_cast<hipStream_t>(stream_of(a[7]));
    lapis::HostSum *sum = nullptr;
    check(is_f64(x) ? lapis::axpby_dot_start<double>(len, ca, (const double *)x.address, cb, (const double *)y.address,
                                                     (double *)d.address, (const double *)z.address, init, st, &sum)
                    : lapis::axpby_dot_start<float>(len, (float)ca, (const float *)x.address, (float)cb, (const float *)y.address,
                                                    (float *)d.address, (const float *)z.address, init, st, &sum));
    return sum_capsule(sum);
  });
}

// (capsule) -> float
LAPIS_PY(py_dot_finish) {
  return guarded([&] {
    arguments("dot_finish", n, 1);
    auto *sum = static_cast<lapis::HostSum *>(PyCapsule_GetPointer(a[0], kSumName));
    if (!sum || PyCapsule_SetDestructor(a[0], nullptr) != 0 || PyCapsule_SetName(a[0], "lapis_hip.finished") != 0) throw Raised();
    double total = 0.0;
    int status;
    Py_BEGIN_ALLOW_THREADS;
    status = lapis::dot_finish(sum, &total);
    Py_END_ALLOW_THREADS;
    check(status);
    return PyFloat_FromDouble(total);
  });
}

// ---- host arrays on their way to the device and back (staging.hpp) ----

struct HostArray {
  Py_buffer view{};
  bool held = false;
  HostArray(PyObject *o, bool writable) {
    if (PyObject_GetBuffer(o, &view, PyBUF_C_CONTIGUOUS | PyBUF_FORMAT | (writable ? PyBUF_WRITABLE : 0)) != 0) throw Raised();
    held = true;
  }
  HostArray(HostArray &&other) noexcept : view(other.view), held(other.held) { other.held = false; }
  ~HostArray() {
    if (held) PyBuffer_Release(&view);
  }
  at::ScalarType type() const {
    const char f = view.format ? view.format[0] : 0;
    if (f == 'd') return at::kDouble;
    if (f == 'f') return at::kFloat;
    if (f == 'i') return at::kInt;
    if (f == 'l' || f == 'q') return at::kLong;
    raise(PyExc_TypeError, "an array of format %s", view.format ? view.format : "?");
  }
};

constexpr const char *kStagedName = "lapis_hip.staged";
typedef std::shared_ptr<lapis::HostOperands> Staged;
void drop_staged(PyObject *capsule) { delete static_cast<Staged *>(PyCapsule_GetPointer(capsule, kStagedName)); }

// (list of arrays, None or (index of positions, index of coordinates, rows, columns), stream)
//   -> (list of tensors, capsule for staged_plan)
LAPIS_PY(py_stage) {
  return guarded([&] {
    arguments("stage", n, 3);
    PyObject *seq = PySequence_Fast(a[0], "stage: a sequence of arrays");
    if (!seq) throw Raised();
    std::unique_ptr<PyObject, void (*)(PyObject *)> seq_guard(seq, [](PyObject *o) { Py_DECREF(o); });
    long long csr[4] = {-1, -1, 0, 0};
    if (a[1] != Py_None && !PyArg_ParseTuple(a[1], "LLLL", &csr[0], &csr[1], &csr[2], &csr[3])) throw Raised();
    std::vector<HostArray> arrays;
    const Py_ssize_t count = PySequence_Fast_GET_SIZE(seq);
    arrays.reserve((size_t)count);
    for (Py_ssize_t i = 0; i < count; ++i) arrays.emplace_back(PySequence_Fast_GET_ITEM(seq, i), false);
    const hipStream_t st = static_cast<hipStream_t>(stream_of(a[2]));
    auto ops = std::make_shared<lapis::HostOperands>();
    ops->use_stream(st);
    if (csr[0] >= 0) {
      if (csr[0] >= count || csr[1] < 0 || csr[1] >= count || arrays[(size_t)csr[0]].type() != at::kInt ||
          arrays[(size_t)csr[1]].type() != at::kInt || arrays[(size_t)csr[0]].view.len != 4 * (csr[2] + 1) || csr[2] < 0 || csr[3] < 0)
        raise(PyExc_ValueError, "stage: a CSR structure of %lld rows", csr[2]);
    }
    for (Py_ssize_t i = 0; i < count; ++i) {
      const Py_buffer &v = arrays[(size_t)i].view;
      if (i == csr[0])
        ops->add_positions(static_cast<const int32_t *>(v.buf), csr[2], arrays[(size_t)csr[1]].view.len / 4);
      else if (i == csr[1])
        ops->add_coordinates(static_cast<const int32_t *>(v.buf), v.len / 4, csr[3]);
      else
        ops->add(v.buf, (size_t)v.len);
    }
    int status;
    Py_BEGIN_ALLOW_THREADS;
    status = ops->upload();
    Py_END_ALLOW_THREADS;
    check(status);
    PyObject *tensors = PyList_New(count);
    if (!tensors) throw Raised();
    const at::Device device(at::kCUDA, c10::hip::getCurrentHIPStream().device_index());
    for (Py_ssize_t i = 0; i < count; ++i) {
      const HostArray &h = arrays[(size_t)i];
      std::vector<int64_t> sizes(h.view.shape, h.view.shape + h.view.ndim);
      const auto options = at::TensorOptions().dtype(h.type()).device(device);
      at::Tensor t = h.view.len == 0 ? at::empty(sizes, options)
                                     : at::from_blob(ops->at<void>((int)i), sizes, [ops](void *) {}, options, device);
      PyList_SET_ITEM(tensors, i, THPVariable_Wrap(std::move(t)));
    }
    PyObject *capsule = PyCapsule_New(new Staged(ops), kStagedName, drop_staged);
    return Py_BuildValue("(NN)", tensors, capsule);
  });
}

// (capsule, index of positions, index of coordinates, bytes per value) -> address of a plan
LAPIS_PY(py_staged_plan) {
  return guarded([&] {
    arguments("staged_plan", n, 4);
    auto *staged = static_cast<Staged *>(PyCapsule_GetPointer(a[0], kStagedName));
    if (!staged) throw Raised();
    lapis_hip_csr_plan *plan = nullptr;
    check((*staged)->create_plan((int)integer(a[1]), (int)integer(a[2]), (int)integer(a[3]), &plan));
    return PyLong_FromVoidPtr(plan);
  });
}

// (tensor, array, stream): the array gets the tensor's elements, after what is queued on the stream
LAPIS_PY(py_fetch) {
  return guarded([&] {
    arguments("fetch", n, 3);
    const Operand t = operand(a[0]);
    HostArray to(a[1], true);
    if (!t.tensor || !t.tensor->is_contiguous() || (int64_t)t.tensor->nbytes() != (int64_t)to.view.len)
      raise(PyExc_ValueError, "fetch: %lld bytes of a contiguous tensor", (long long)to.view.len);
    lapis::HostOperands ops;
    ops.use_stream(static_cast<hipStream_t>(stream_of(a[2])));
    int status;
    Py_BEGIN_ALLOW_THREADS;
    status = ops.upload();
    if (status == LAPIS_HIP_OK) status = ops.download(t.address, (size_t)to.view.len, to.view.buf);
    Py_END_ALLOW_THREADS;
    check(status);
    return give(a[1]);
  });
}

// (a, x, b, y, dst, stream): dst = a x + b y
LAPIS_PY(py_axpby) {
  return guarded([&] {
    arguments("axpby", n, 6);
    const double ca = number(a[0]), cb = number(a[2]);
    const Operand x = operand(a[1]), y = operand(a[3]), d = operand(a[4]);
    const int64_t len = length("axpby", x);
    holds("axpby", len, x, x.tensor);
    holds("axpby", len, y, x.tensor);
    holds("axpby", len, d, x.tensor);
    if (is_f64(x))
      check(lapis_hip_axpby_f64(len, ca, (const double *)x.address, cb, (const double *)y.address, (double *)d.address, stream_of(a[5])));
    else
      check(lapis_hip_axpby_f32(len, (float)ca, (const float *)x.address, (float)cb, (const float *)y.address, (float *)d.address,
                                stream_of(a[5])));
    return give(a[4]);
  });
}

// (x, y, dst, stream)
template <int (*F64)(int64_t, const double *, const double *, double *, lapis_hip_stream_t),
          int (*F32)(int64_t, const float *, const float *, float *, lapis_hip_stream_t)>
PyObject *two_operands(const char *what, PyObject *const *a, Py_ssize_t n) {
  return guarded([&] {
    arguments(what, n, 4);
    const Operand x = operand(a[0]), y = operand(a[1]), d = operand(a[2]);
    const int64_t len = length(what, x);
    holds(what, len, x, x.tensor);
    holds(what, len, y, x.tensor);
    holds(what, len, d, x.tensor);
    if (is_f64(x))
      check(F64(len, (const double *)x.address, (const double *)y.address, (double *)d.address, stream_of(a[3])));
    else
      check(F32(len, (const float *)x.address, (const float *)y.address, (float *)d.address, stream_of(a[3])));
    return give(a[2]);
  });
}
LAPIS_PY(py_mult) { return two_operands<lapis_hip_mult_f64, lapis_hip_mult_f32>("mult", a, n); }
LAPIS_PY(py_div) { return two_operands<lapis_hip_div_f64, lapis_hip_div_f32>("div", a, n); }

// (dst, value, stream)
LAPIS_PY(py_fill) {
  return guarded([&] {
    arguments("fill", n, 3);
    const Operand d = operand(a[0]);
    const int64_t len = length("fill", d);
    const double v = number(a[1]);
    if (is_f64(d)) check(lapis_hip_fill_f64(len, v, (double *)d.address, stream_of(a[2])));
    else check(lapis_hip_fill_f32(len, (float)v, (float *)d.address, stream_of(a[2])));
    return give(a[0]);
  });
}

// (src, dst, stream)
LAPIS_PY(py_copy) {
  return guarded([&] {
    arguments("copy", n, 3);
    const Operand s = operand(a[0]), d = operand(a[1]);
    const int64_t len = length("copy", s);
    holds("copy", len, s, s.tensor);
    holds("copy", len, d, s.tensor);
    if (is_f64(s)) check(lapis_hip_copy_f64(len, (const double *)s.address, (double *)d.address, stream_of(a[2])));
    else check(lapis_hip_copy_f32(len, (const float *)s.address, (float *)d.address, stream_of(a[2])));
    return give(a[1]);
  });
}

// (plan, n, pos, crd, val, b, dinv, tol, maxiter, x, work, stream) -> (iterations, relative residual)
LAPIS_PY(py_pcg) {
  return guarded([&] {
    arguments("pcg", n, 12);
    const int64_t rows = integer(a[1]);
    const Operand pos = operand(a[2]), crd = operand(a[3]), val = operand(a[4]), b = operand(a[5]), dinv = operand(a[6]),
                  x = operand(a[9]), work = operand(a[10]);
    indices("pcg", pos);
    indices("pcg", crd);
    holds("pcg", rows + 1, pos);
    holds("pcg", rows, b, val.tensor);
    holds("pcg", rows, dinv, val.tensor);
    holds("pcg", rows, x, val.tensor);
    holds("pcg", 4 * rows, work, val.tensor);
    if (crd.tensor) holds("pcg", crd.tensor->numel(), val);
    for (const Operand *o : {&val, &b, &dinv, &x, &work})
      if (o->tensor && o->tensor->scalar_type() != at::kDouble)
        raise(PyExc_TypeError, "pcg: operands are float64, got %s", type_name(o->tensor->scalar_type()));
    const double tol = number(a[7]);
    const int64_t maxiter = integer(a[8]);
    lapis_hip_csr_plan *plan = plan_of(a[0]);
    const lapis_hip_stream_t st = stream_of(a[11]);
    uint64_t iters = 0;
    double relres = 0.0;
    int status;
    Py_BEGIN_ALLOW_THREADS;
    status = lapis_hip_pcg_f64_i32(plan, rows, (const int32_t *)pos.address, (const int32_t *)crd.address,
                                   (const double *)val.address, (const double *)b.address, (const double *)dinv.address, tol,
                                   (uint64_t)maxiter, (double *)x.address, &iters, &relres, (double *)work.address, st);
    Py_END_ALLOW_THREADS;
    check(status);
    return Py_BuildValue("(Kd)", (unsigned long long)iters, relres);
  });
}

// setup(check, init)
PyObject *py_setup(PyObject *, PyObject *args) {
  PyObject *check_fn, *init_fn;
  if (!PyArg_ParseTuple(args, "OO", &check_fn, &init_fn)) return nullptr;
  Py_INCREF(check_fn);
  Py_XSETREF(g_check, check_fn);
  Py_INCREF(init_fn);
  Py_XSETREF(g_init, init_fn);
  Py_RETURN_NONE;
}

#define LAPIS_METHOD(name) {#name, (PyCFunction)(void (*)(void))py_##name, METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {LAPIS_METHOD(spmv), LAPIS_METHOD(spmm), LAPIS_METHOD(bspmm_csrv), LAPIS_METHOD(dot),
                           LAPIS_METHOD(dot_host), LAPIS_METHOD(axpby), LAPIS_METHOD(mult), LAPIS_METHOD(div),
                           LAPIS_METHOD(fill), LAPIS_METHOD(copy), LAPIS_METHOD(pcg), LAPIS_METHOD(spmv_overwrite),
                           LAPIS_METHOD(spmv_dot_start), LAPIS_METHOD(dot_start), LAPIS_METHOD(axpby_dot_start),
                           LAPIS_METHOD(dot_finish), LAPIS_METHOD(stage), LAPIS_METHOD(staged_plan), LAPIS_METHOD(fetch),
                           {"setup", py_setup, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_lapis_calls", "Device-resident calls of the gfx950 kernel library.", -1,
                        g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__lapis_calls(void) { return PyModule_Create(&g_module); }
