// The operators of cobalt_amd/ops.py as a CPython extension: argument checks, output and scratch
// allocation and the call into libcbk_hip.so.
//
// Why native: a decode call is one or two kernels of 5 to 20 us.  Through ctypes (descriptor built
// field by field, workspace looked up, a dozen conversions) the host needed 16.7 us for one
// CobaltLinear call of a 1024 x 4096 matrix at one row, three times its kernel, and about 20 us per
// gemv_batch: eager decode ran at the speed of the interpreter.
//
// Scratch comes from torch's caching allocator on every call (about a microsecond, stream-ordered,
// private to the graph when the call is captured) instead of a buffer kept per stream: calls from
// several threads on one stream cannot meet in it, and it goes back when the call has been enqueued.
#include <Python.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <ATen/EmptyTensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/InlineDeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <memory>
#include "cbk_internal.h"

namespace {

PyObject* g_error = nullptr;                                        // cobalt_amd._lib.CbkError

// One packed matrix: the image and where its arrays are in it.  The addresses are formed per
// call, so a tensor whose storage is exchanged (module.to()) is followed, and so is a change inside
// the two containers the Python object owns: the offsets and the row ranges are read from them
// every time (seven lookups, 0.1 us).
struct Matrix {
  PyObject_HEAD
  at::Tensor* blob;
  PyObject* offs;                                                   // dict: byte offset of every array in the image
  PyObject* splits;                                                 // sequence: cs_split0, cs_split1
  cbk_desc d;
};

PyObject* g_key[5];                                                 // "data", "row_off", "scale", "zero", "col_scale"

void matrix_dealloc(PyObject* o) {
  Matrix* m = (Matrix*)o;
  delete m->blob;
  Py_XDECREF(m->offs);
  Py_XDECREF(m->splits);
  Py_TYPE(o)->tp_free(o);
}

PyObject* matrix_new(PyTypeObject* t, PyObject* args, PyObject*) {
  PyObject *blob, *offs, *splits, *ints;
  if (!PyArg_ParseTuple(args, "OO!OO!", &blob, &PyDict_Type, &offs, &splits, &PyTuple_Type, &ints)) return nullptr;
  if (!THPVariable_Check(blob) || PyTuple_GET_SIZE(ints) != 8) {
    PyErr_SetString(PyExc_TypeError, "Matrix(blob tensor, offsets, row ranges, 8 integers)");
    return nullptr;
  }
  Matrix* m = (Matrix*)t->tp_alloc(t, 0);
  if (!m) return nullptr;
  m->blob = new at::Tensor(THPVariable_Unpack(blob));
  Py_INCREF(offs); m->offs = offs;
  Py_INCREF(splits); m->splits = splits;
  long long v[8];
  for (int i = 0; i < 8; ++i) v[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(ints, i));
  if (PyErr_Occurred()) { Py_DECREF(m); return nullptr; }
  m->d = cbk_desc{};
  m->d.K = (int32_t)v[0]; m->d.N = (int32_t)v[1]; m->d.layout = (int32_t)v[2]; m->d.bits = (int32_t)v[3];
  m->d.group = (int32_t)v[4]; m->d.keep = (int32_t)v[5]; m->d.cs_rows = (int32_t)v[6]; m->d.flags = (int32_t)v[7];
  return (PyObject*)m;
}

PyTypeObject MatrixType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// Other Python threads run while this one allocates and launches: a launch waits when its queue is full, an allocation
// may wait for the device.  No Python object is touched and no Python exception set in its scope.
struct GilRelease {
  PyThreadState* s = PyEval_SaveThread();
  ~GilRelease() { PyEval_RestoreThread(s); }
};

struct Fail {};                                                     // a Python exception has been set

[[noreturn]] void fail(PyObject* type, const std::string& msg) {
  PyErr_SetString(type, msg.c_str());
  throw Fail{};
}

void check(int rc, const char* what) {
  if (rc) fail(g_error, std::string(what) + " failed: " + cbk_strerror(rc) + " (status " + std::to_string(rc) + ")");
}

// Holds the interpreter lock.
cbk_desc desc_of(const Matrix* m) {
  cbk_desc d = m->d;
  const uint8_t* base = (const uint8_t*)m->blob->const_data_ptr();
  const void* p[5];
  for (int i = 0; i < 5; ++i) {
    PyObject* o = i == 4 && !d.cs_rows ? nullptr : PyDict_GetItemWithError(m->offs, g_key[i]);
    if (!o) {
      if (PyErr_Occurred()) throw Fail{};
      if (i != 1 && !(i == 4 && !d.cs_rows)) { PyErr_SetObject(PyExc_KeyError, g_key[i]); throw Fail{}; }
      p[i] = nullptr;
      continue;
    }
    const long long off = PyLong_AsLongLong(o);
    if (off == -1 && PyErr_Occurred()) throw Fail{};
    p[i] = base + off;
  }
  d.data = p[0]; d.row_off = p[1]; d.scale = p[2]; d.zero = p[3]; d.col_scale = p[4];
  for (int i = 0; i < 2; ++i) {
    PyObject* o = PySequence_GetItem(m->splits, i);
    if (!o) throw Fail{};
    const long long v = PyLong_AsLongLong(o);
    Py_DECREF(o);
    if (v == -1 && PyErr_Occurred()) throw Fail{};
    (i ? d.cs_split1 : d.cs_split0) = (int32_t)v;
  }
  return d;
}

const Matrix* as_matrix(PyObject* o) {
  if (Py_TYPE(o) != &MatrixType) fail(PyExc_TypeError, "a native matrix handle is expected");
  return (const Matrix*)o;
}

// None -> undefined tensor
at::Tensor as_tensor(PyObject* o, const char* what) {
  if (o == Py_None) return at::Tensor();
  if (!THPVariable_Check(o)) fail(PyExc_TypeError, std::string(what) + " must be a tensor");
  return THPVariable_Unpack(o);
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return CBK_F32;
    case at::kHalf: return CBK_F16;
    case at::kBFloat16: return CBK_BF16T;
    default:
      fail(PyExc_TypeError, std::string("unsupported dtype ") + c10::toString(t) +
                                "; the layer takes float16 / bfloat16 activations");
  }
}

at::ScalarType out_type(PyObject* o, const at::Tensor& x) {
  if (o == Py_None) return x.scalar_type();
  if (!THPDtype_Check(o)) fail(PyExc_TypeError, "out_dtype must be a torch.dtype");
  return ((THPDtype*)o)->scalar_type;
}

void require_gpu(const Matrix* m, const at::Tensor& x, const at::Tensor& bias) {
  if (!m->blob->is_cuda())
    fail(g_error, "the packed matrix must live on the GPU (PackedMatrix.to('cuda')); this package has no CPU execution path");
  for (const at::Tensor* t : {&x, &bias})
    if (t->defined() && t->device() != m->blob->device())
      fail(g_error, "tensor on " + t->device().str() + ", packed matrix on " + m->blob->device().str());
}

void check_features(const at::Tensor& x, int64_t N) {
  if (x.dim() < 1 || x.size(-1) != N)
    fail(PyExc_ValueError, "x has " + std::to_string(x.dim() ? x.size(-1) : 1) + " input features, the matrix has N=" + std::to_string(N));
}
// x as [M, N] rows of unit stride the kernels can read with 16-byte loads (a copy if it is not)
struct Rows { at::Tensor keep; const void* p; int64_t M, ld; };
Rows rows_of(const at::Tensor& x, int64_t N) {
  Rows r;
  r.M = x.numel() / N;
  const bool flat = x.is_contiguous();
  if (flat || (x.dim() == 2 && x.stride(1) == 1 && x.stride(0) % 8 == 0 && x.stride(0) >= N)) {
    r.p = x.const_data_ptr();
    r.ld = flat || r.M <= 1 ? N : x.stride(0);
    if (((uintptr_t)r.p & 15) == 0) return r;
  }
  at::Tensor t = x.reshape({-1, N});
  if (t.stride(1) != 1 || (t.size(0) > 1 && (t.stride(0) % 8 || t.stride(0) < N)) || ((uintptr_t)t.const_data_ptr() & 15))
    t = t.clone(at::MemoryFormat::Contiguous);
  r.keep = t;
  r.p = t.const_data_ptr();
  r.ld = r.M > 1 ? t.stride(0) : N;
  return r;
}

at::Tensor out_for(const at::Tensor& x, int64_t K, at::ScalarType dt) {
  c10::SmallVector<int64_t, 6> shape(x.sizes().begin(), x.sizes().end());
  shape.back() = K;
  return at::empty(shape, x.options().dtype(dt).requires_grad(false).memory_format(at::MemoryFormat::Contiguous));
}

at::Tensor scratch(const at::Tensor& like, size_t bytes) {
  return bytes ? at::empty({(int64_t)bytes}, like.options().dtype(at::kByte)) : at::Tensor();
}

void* stream_of(const at::Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

template <class F>
PyObject* guarded(F&& f) {
  HANDLE_TH_ERRORS
  try {
    at::AutoDispatchBelowADInplaceOrView no_autograd;
    return f();
  } catch (const Fail&) {
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

bool arity(Py_ssize_t n, Py_ssize_t want) {
  if (n == want) return true;
  PyErr_SetString(PyExc_TypeError, "wrong number of arguments");
  return false;
}

// matmul(entry 0 gemv / 1 gemm / 2 linear, matrix, x, bias, out_dtype, workspace) -> y
PyObject* py_matmul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!arity(n, 6)) return nullptr;
  return guarded([&]() -> PyObject* {
    const long entry = PyLong_AsLong(a[0]);
    const Matrix* m = as_matrix(a[1]);
    const at::Tensor x = as_tensor(a[2], "x");
    at::Tensor bias = as_tensor(a[3], "bias");
    at::Tensor ws = as_tensor(a[5], "workspace");
    if (!x.defined()) fail(PyExc_TypeError, "x must be a tensor");
    require_gpu(m, x, bias);
    const cbk_desc d = desc_of(m);
    check_features(x, d.N);
    const at::ScalarType odt = out_type(a[4], x);
    const bool any = x.numel() > 0;
    const int xdt = any ? dtype_code(x.scalar_type()) : 0, ydt = any ? dtype_code(odt) : 0;
    at::Tensor y;
    int rc = CBK_OK;
    {
      const GilRelease other_threads_run;
      y = out_for(x, d.K, odt);
      if (any) {
        const Rows r = rows_of(x, d.N);
        const int M = (int)r.M;
        if (bias.defined() && bias.scalar_type() != odt) bias = bias.to(odt);
        const c10::DeviceGuard guard(x.device());
        if (!ws.defined())
          ws = scratch(x, entry == 0 || (entry == 2 && M <= 8) ? cbk::decode_workspace_bytes(&d, M) : cbk_workspace_bytes(&d, M));
        auto fn = entry == 0 ? cbk_gemv : entry == 1 ? cbk_gemm : cbk_linear;
        rc = fn(&d, r.p, xdt, M, r.ld, y.mutable_data_ptr(), ydt, d.K, bias.defined() ? bias.const_data_ptr() : nullptr,
                ws.defined() ? ws.mutable_data_ptr() : nullptr, ws.defined() ? ws.nbytes() : 0, stream_of(x));
      }
    }
    check(rc, entry == 0 ? "cbk_gemv" : entry == 1 ? "cbk_gemm" : "cbk_linear");
    return THPVariable_Wrap(y);
  });
}

// linear_act(matrix, x, act, bias, out_dtype) -> y
PyObject* py_linear_act(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!arity(n, 5)) return nullptr;
  return guarded([&]() -> PyObject* {
    const Matrix* m = as_matrix(a[0]);
    const at::Tensor x = as_tensor(a[1], "x");
    const int act = (int)PyLong_AsLong(a[2]);
    at::Tensor bias = as_tensor(a[3], "bias");
    if (!x.defined()) fail(PyExc_TypeError, "x must be a tensor");
    require_gpu(m, x, bias);
    const cbk_desc d = desc_of(m);
    check_features(x, d.N);
    if (d.K % 2) fail(PyExc_ValueError, "a gate/up matrix has an even number of rows");
    const at::ScalarType odt = out_type(a[4], x);
    const bool any = x.numel() > 0;
    const int xdt = any ? dtype_code(x.scalar_type()) : 0, ydt = any ? dtype_code(odt) : 0;
    at::Tensor y;
    int rc = CBK_OK;
    {
      const GilRelease other_threads_run;
      y = out_for(x, d.K / 2, odt);
      if (any) {
        const Rows r = rows_of(x, d.N);
        const int M = (int)r.M;
        if (bias.defined() && bias.scalar_type() != odt) bias = bias.to(odt);
        const c10::DeviceGuard guard(x.device());
        const at::Tensor ws = scratch(x, cbk_linear_act_workspace_bytes(&d, M, ydt));
        rc = cbk_linear_act(&d, r.p, xdt, M, r.ld, y.mutable_data_ptr(), ydt, d.K / 2,
                            bias.defined() ? bias.const_data_ptr() : nullptr, act,
                            ws.defined() ? ws.mutable_data_ptr() : nullptr, ws.defined() ? ws.nbytes() : 0, stream_of(x));
      }
    }
    check(rc, "cbk_linear_act");
    return THPVariable_Wrap(y);
  });
}

// what a decode call of the matrices launches; see cbk::decode_choice
cbk::DecodeChoice choice_of(PyObject* const* a, bool room) {
  if (!PyList_Check(a[0]) || PyList_GET_SIZE(a[0]) < 1 || PyList_GET_SIZE(a[0]) > 8)
    fail(PyExc_TypeError, "a list of one to eight matrices is expected");
  const int k = (int)PyList_GET_SIZE(a[0]);
  cbk_desc d[8];
  for (int i = 0; i < k; ++i) d[i] = desc_of(as_matrix(PyList_GET_ITEM(a[0], i)));
  const long M = PyLong_AsLong(a[1]);
  if (PyErr_Occurred()) throw Fail{};
  cbk::DecodeChoice c;
  check(cbk::decode_choice(k, d, (int)M, room, &c), "cbk::decode_choice");
  return c;
}
// decode_choice([matrix], M) -> (table of the main kernel, its slots, table of the split kernel)
PyObject* py_decode_choice(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!arity(n, 2)) return nullptr;
  return guarded([&]() -> PyObject* {
    const cbk::DecodeChoice c = choice_of(a, true);
    return Py_BuildValue("iii", c.main_table, c.main_slots, c.split_table);
  });
}
// decode_slabs([matrix], M) -> column slabs a row is staged in where there is no workspace (1: whole)
PyObject* py_decode_slabs(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!arity(n, 2)) return nullptr;
  return guarded([&]() -> PyObject* { return PyLong_FromLong(choice_of(a, false).main_slabs); });
}

// gemm_plan(matrix, M, act or -1) -> (kernel, ti, nsplit); see cbk::gemm_choice
PyObject* py_gemm_plan(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!arity(n, 3)) return nullptr;
  return guarded([&]() -> PyObject* {
    const cbk_desc d = desc_of(as_matrix(a[0]));
    const long M = PyLong_AsLong(a[1]), act = PyLong_AsLong(a[2]);
    if (PyErr_Occurred()) throw Fail{};
    const cbk::GemmChoice c = cbk::gemm_choice(&d, (int)M, (int)act);
    return Py_BuildValue("iii", c.kernel, c.ti, c.nsplit);
  });
}

// gemm_last_round(matrix, M, kernel, ti, nsplit) -> (row tiles, ti); see cbk::gemm_last_round
PyObject* py_gemm_last_round(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!arity(n, 5)) return nullptr;
  return guarded([&]() -> PyObject* {
    const cbk_desc d = desc_of(as_matrix(a[0]));
    const long M = PyLong_AsLong(a[1]);
    const cbk::GemmChoice c{(int)PyLong_AsLong(a[2]), (int)PyLong_AsLong(a[3]), (int)PyLong_AsLong(a[4])};
    if (PyErr_Occurred()) throw Fail{};
    int rows, ti;
    cbk::gemm_last_round(&d, (int)M, c, &rows, &ti);
    return Py_BuildValue("ii", rows, ti);
  });
}

// gemm_column_parts(matrix, M, kernel, ti, nsplit) -> (parts, stages of the first, of a further one); see cbk::gemm_column_parts
PyObject* py_gemm_column_parts(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!arity(n, 5)) return nullptr;
  return guarded([&]() -> PyObject* {
    const cbk_desc d = desc_of(as_matrix(a[0]));
    const long M = PyLong_AsLong(a[1]);
    const cbk::GemmChoice c{(int)PyLong_AsLong(a[2]), (int)PyLong_AsLong(a[3]), (int)PyLong_AsLong(a[4])};
    if (PyErr_Occurred()) throw Fail{};
    int parts, first, rest;
    cbk::gemm_column_parts(&d, (int)M, c, &parts, &first, &rest);
    return Py_BuildValue("iii", parts, first, rest);
  });
}

// gemm_as(matrix, x, bias, out_dtype, kernel, ti, nsplit, act or -1) -> y; see cbk::gemm_as
PyObject* py_gemm_as(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!arity(n, 8)) return nullptr;
  return guarded([&]() -> PyObject* {
    const Matrix* m = as_matrix(a[0]);
    const at::Tensor x = as_tensor(a[1], "x"), bias = as_tensor(a[2], "bias");
    if (!x.defined() || !x.numel()) fail(PyExc_TypeError, "x must be a tensor with elements");
    require_gpu(m, x, bias);
    const cbk_desc d = desc_of(m);
    check_features(x, d.N);
    const at::ScalarType odt = out_type(a[3], x);
    const int xdt = dtype_code(x.scalar_type()), ydt = dtype_code(odt);
    const cbk::GemmChoice c{(int)PyLong_AsLong(a[4]), (int)PyLong_AsLong(a[5]), (int)PyLong_AsLong(a[6])};
    const int act = (int)PyLong_AsLong(a[7]), Ko = act >= 0 ? d.K / 2 : d.K;
    if (PyErr_Occurred()) throw Fail{};
    if (bias.defined() && bias.scalar_type() != odt) fail(PyExc_TypeError, "the bias must have the output's type");
    at::Tensor y;
    int rc = CBK_OK;
    {
      const GilRelease other_threads_run;
      const Rows r = rows_of(x, d.N);
      y = out_for(x, Ko, odt);
      const c10::DeviceGuard guard(x.device());
      const at::Tensor ws = scratch(x, cbk::gemm_as_workspace_bytes(&d, (int)r.M, c, act, ydt));
      rc = cbk::gemm_as(&d, c, r.p, xdt, (int)r.M, r.ld, y.mutable_data_ptr(), ydt, Ko,
                        bias.defined() ? bias.const_data_ptr() : nullptr, act, ws.defined() ? ws.mutable_data_ptr() : nullptr,
                        ws.defined() ? ws.nbytes() : 0, stream_of(x));
    }
    check(rc, "cbk::gemm_as");
    return THPVariable_Wrap(y);
  });
}

// dequant(matrix, dtype, row0, nrows, with_col_scale) -> W_hat[row0 : row0 + nrows]
PyObject* py_dequant(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!arity(n, 5)) return nullptr;
  return guarded([&]() -> PyObject* {
    const Matrix* m = as_matrix(a[0]);
    require_gpu(m, at::Tensor(), at::Tensor());
    if (!THPDtype_Check(a[1])) fail(PyExc_TypeError, "dtype must be a torch.dtype");
    const at::ScalarType dt = ((THPDtype*)a[1])->scalar_type;
    const long long row0 = PyLong_AsLongLong(a[2]), nrows = PyLong_AsLongLong(a[3]);
    const int cs = PyObject_IsTrue(a[4]);
    if (PyErr_Occurred()) throw Fail{};
    const cbk_desc d = desc_of(m);
    const int odt = dtype_code(dt);
    const at::TensorOptions like = m->blob->options().dtype(dt);
    at::Tensor out;
    int rc = CBK_OK;
    {
      const GilRelease other_threads_run;
      out = at::empty({(int64_t)nrows, (int64_t)d.N}, like);
      const c10::DeviceGuard guard(out.device());
      rc = cbk_dequant(&d, (int)row0, (int)nrows, cs, out.mutable_data_ptr(), odt, d.N, stream_of(out));
    }
    check(rc, "cbk_dequant");
    return THPVariable_Wrap(out);
  });
}

// gemv_batch(list of matrices, list of x, list of biases or None, out_dtype) -> list of y
PyObject* py_gemv_batch(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  if (!arity(nargs, 4)) return nullptr;
  return guarded([&]() -> PyObject* {
    if (!PyList_Check(a[0]) || !PyList_Check(a[1]) || !(a[2] == Py_None || PyList_Check(a[2])))
      fail(PyExc_TypeError, "lists of matrices, activations and biases are expected");
    const Py_ssize_t n = PyList_GET_SIZE(a[0]);
    if (n < 1 || PyList_GET_SIZE(a[1]) < n || (a[2] != Py_None && PyList_GET_SIZE(a[2]) < n))
      fail(PyExc_ValueError, "one activation (and bias) per matrix is expected");
    if (n > 8) check(CBK_ERR_SHAPE, "cbk_gemv_batch");
    cbk_desc d[8];
    at::Tensor x[8], y[8], b[8];
    at::ScalarType odt = at::kHalf;
    for (Py_ssize_t i = 0; i < n; ++i) {
      const Matrix* m = as_matrix(PyList_GET_ITEM(a[0], i));
      x[i] = as_tensor(PyList_GET_ITEM(a[1], i), "x");
      if (!x[i].defined()) fail(PyExc_TypeError, "x must be a tensor");
      if (a[2] != Py_None) b[i] = as_tensor(PyList_GET_ITEM(a[2], i), "bias");
      require_gpu(m, x[i], b[i]);
      d[i] = desc_of(m);
      check_features(x[i], d[i].N);
      if (i == 0) odt = out_type(a[3], x[0]);
      if (x[i].numel() / d[i].N != x[0].numel() / d[0].N || x[i].scalar_type() != x[0].scalar_type())
        fail(PyExc_ValueError, "all activations of a batch share the row count and the dtype");
    }
    const int xdt = dtype_code(x[0].scalar_type()), ydt = dtype_code(odt);
    int rc = CBK_OK;
    {
      const GilRelease other_threads_run;
      Rows r[8];
      const void *xp[8], *bp[8];
      void* yp[8];
      int64_t ldx[8], ldy[8];
      size_t need = 0;
      for (Py_ssize_t i = 0; i < n; ++i) {
        r[i] = rows_of(x[i], d[i].N);
        y[i] = out_for(x[i], d[i].K, odt);
        if (b[i].defined() && b[i].scalar_type() != odt) b[i] = b[i].to(odt);
        xp[i] = r[i].p; ldx[i] = r[i].ld;
        yp[i] = y[i].mutable_data_ptr(); ldy[i] = d[i].K;
        bp[i] = b[i].defined() ? b[i].const_data_ptr() : nullptr;
      }
      need = cbk::decode_batch_workspace_bytes((int)n, d, (int)r[0].M);
      const c10::DeviceGuard guard(x[0].device());
      const at::Tensor ws = scratch(x[0], need);
      rc = cbk_gemv_batch((int)n, d, xp, ldx, xdt, (int)r[0].M, yp, ldy, ydt, bp,
                          ws.defined() ? ws.mutable_data_ptr() : nullptr, need, stream_of(x[0]));
    }
    check(rc, "cbk_gemv_batch");
    PyObject* out = PyList_New(n);
    if (!out) throw Fail{};
    for (Py_ssize_t i = 0; i < n; ++i) PyList_SET_ITEM(out, i, THPVariable_Wrap(y[i]));
    return out;
  });
}

// pack_begin(mask or None, q, scale, zero, col_scale or None, layout, bits, group, keep, fix_zero, tiled) ->
//   (blob, offsets of data / scale / zero / col_scale (-1: none), cs_rows, data_bytes, pending)
// pack_end(pending) -> (status, groups re-derived, largest zero point, survivors in the mask)
// The caller has checked shapes and devices.  One kernel writes every byte of the image, and its figures
// to pinned memory, 16 bytes a workgroup (a copy of them behind the kernel is a second dependent piece of work for the
// stream: 14336 x 4096 51.8 -> 48.8 us).  pack_end waits for the stream: what the caller does in between costs
// no time.
struct PendingPack {                                                // holds the memory the kernel writes to until it has ended
  at::Tensor host;
  c10::hip::HIPStream stream;
  bool done = false;
  PendingPack(at::Tensor h, c10::hip::HIPStream s) : host(std::move(h)), stream(s) {}
  ~PendingPack() {                                                  // not done: dropped without pack_end
    if (!done) try { stream.synchronize(); } catch (...) {}
  }
};
constexpr const char* PENDING = "cobalt_amd.pending_pack";
void pending_free(PyObject* o) { delete (PendingPack*)PyCapsule_GetPointer(o, PENDING); }

PyObject* py_pack_begin(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!arity(n, 11)) return nullptr;
  return guarded([&]() -> PyObject* {
    at::Tensor mask = as_tensor(a[0], "mask"), q = as_tensor(a[1], "q"), scale = as_tensor(a[2], "scale"),
               zero = as_tensor(a[3], "zero"), cs = as_tensor(a[4], "col_scale");
    cbk_desc d{};
    d.layout = (int)PyLong_AsLong(a[5]); d.bits = (int)PyLong_AsLong(a[6]);
    d.group = (int)PyLong_AsLong(a[7]); d.keep = (int)PyLong_AsLong(a[8]);
    const bool fix = PyObject_IsTrue(a[9]), tiled = PyObject_IsTrue(a[10]);
    if (PyErr_Occurred()) throw Fail{};
    const int64_t K = q.size(0), N = q.size(1), G = N / d.group, kr = tiled ? (K + 15) / 16 * 16 : K;
    int64_t cs_rows = 0, off[4] = {0, 0, 0, -1}, stride = 0;
    at::Tensor blob;
    std::unique_ptr<PendingPack> pending;
    int rc = CBK_OK;
    {
      const GilRelease other_threads_run;
      const at::Device dev = q.device();
      const c10::DeviceGuard guard(dev);
      d.K = (int32_t)K; d.N = (int32_t)N; d.flags = tiled ? CBK_FLAG_TILED16 : 0;
      q = (q.scalar_type() == at::kByte ? q : q.clamp(0, 255).to(at::kByte)).contiguous();
      if (mask.defined()) mask = mask.to(dev).reshape({K, N / 8}).contiguous();
      scale = scale.to(dev, at::kHalf).reshape({K, G}).contiguous();
      zero = zero.to(dev).reshape({K, G});
      zero = (zero.scalar_type() == at::kByte ? zero : zero.to(at::kHalf)).contiguous();
      if (cs.defined()) {
        cs = cs.to(dev, at::kHalf).reshape({-1, N}).contiguous();
        if ((uintptr_t)cs.const_data_ptr() & 15) cs = cs.clone(at::MemoryFormat::Contiguous);
        cs_rows = cs.size(0);
      }
      // the packing kernel reads q with 16-byte and the mask with 4-byte loads
      if ((uintptr_t)q.const_data_ptr() & 15) q = q.clone(at::MemoryFormat::Contiguous);
      if (mask.defined() && ((uintptr_t)mask.const_data_ptr() & 3)) mask = mask.clone(at::MemoryFormat::Contiguous);
      stride = (int64_t)cbk_row_stride(&d);
      const int64_t size[4] = {kr * stride + (tiled ? 512 : 64), kr * G * 2, kr * G, cs_rows * N * 2};
      const int na = cs_rows ? 4 : 3;
      int64_t pos = 0;
      cbk::PackExtra x{};
      for (int i = 0; i < na; ++i) { off[i] = pos; pos = (pos + size[i] + 255) / 256 * 256; }
      const at::TensorOptions bytes = at::TensorOptions().dtype(at::kByte).device(dev);
      blob = at::empty({pos}, bytes);
      uint8_t* base = (uint8_t*)blob.mutable_data_ptr();
      for (int i = 0; i < na; ++i) {
        x.gap[i] = base + off[i] + size[i];
        x.gap_bytes[i] = (uint32_t)((i + 1 < na ? off[i + 1] : pos) - off[i] - size[i]);
      }
      d.data = base + off[0]; d.scale = base + off[1]; d.zero = base + off[2];
      if (cs_rows) {
        x.cs_src = cs.const_data_ptr(); x.cs_dst = base + off[3]; x.cs_units = (uint32_t)(size[3] / 16);
      }
      pending.reset(new PendingPack(at::empty({cbk::pack_records(K, N), 4}, at::TensorOptions().dtype(at::kInt).pinned_memory(true)),
                                    c10::hip::getCurrentHIPStream(dev.index())));
      x.counts = (uint32_t*)pending->host.mutable_data_ptr();
      rc = cbk::pack_image(&d, mask.defined() ? mask.const_data_ptr() : nullptr, q.const_data_ptr(), scale.const_data_ptr(),
                           zero.const_data_ptr(), zero.scalar_type() == at::kByte ? CBK_U8 : CBK_F16, fix ? 1 : 0, nullptr, &x,
                           pending->stream.stream());
    }
    check(rc, "cbk_pack");
    PyObject* const capsule = PyCapsule_New(pending.get(), PENDING, pending_free);
    if (!capsule) throw Fail{};
    pending.release();
    return Py_BuildValue("N(LLLL)LLN", THPVariable_Wrap(blob), (long long)off[0], (long long)off[1], (long long)off[2],
                         (long long)off[3], (long long)cs_rows, (long long)(kr * stride), capsule);
  });
}

PyObject* py_pack_end(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!arity(n, 1)) return nullptr;
  return guarded([&]() -> PyObject* {
    PendingPack* const p = (PendingPack*)PyCapsule_GetPointer(a[0], PENDING);
    if (!p) throw Fail{};
    {
      const GilRelease other_threads_run;
      p->stream.synchronize();
    }
    p->done = true;
    const uint32_t* h = (const uint32_t*)p->host.const_data_ptr();
    uint32_t status = 0, fixed = 0, zmax = 0;
    unsigned long long surv = 0;
    for (int64_t i = 0, n = p->host.size(0); i < n; ++i, h += 4) {
      status |= h[0]; fixed += h[1]; surv += h[3];
      zmax = zmax > h[2] ? zmax : h[2];
    }
    return Py_BuildValue("IIIK", status, fixed, zmax, surv);
  });
}

PyObject* py_set_error(PyObject*, PyObject* e) {
  Py_INCREF(e);
  Py_XSETREF(g_error, e);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"matmul", (PyCFunction)(void (*)())py_matmul, METH_FASTCALL, nullptr},
    {"linear_act", (PyCFunction)(void (*)())py_linear_act, METH_FASTCALL, nullptr},
    {"gemv_batch", (PyCFunction)(void (*)())py_gemv_batch, METH_FASTCALL, nullptr},
    {"decode_choice", (PyCFunction)(void (*)())py_decode_choice, METH_FASTCALL, nullptr},
    {"decode_slabs", (PyCFunction)(void (*)())py_decode_slabs, METH_FASTCALL, nullptr},
    {"gemm_plan", (PyCFunction)(void (*)())py_gemm_plan, METH_FASTCALL, nullptr},
    {"gemm_column_parts", (PyCFunction)(void (*)())py_gemm_column_parts, METH_FASTCALL, nullptr},
    {"gemm_last_round", (PyCFunction)(void (*)())py_gemm_last_round, METH_FASTCALL, nullptr},
    {"gemm_as", (PyCFunction)(void (*)())py_gemm_as, METH_FASTCALL, nullptr},
    {"dequant", (PyCFunction)(void (*)())py_dequant, METH_FASTCALL, nullptr},
    {"pack_begin", (PyCFunction)(void (*)())py_pack_begin, METH_FASTCALL, nullptr},
    {"pack_end", (PyCFunction)(void (*)())py_pack_end, METH_FASTCALL, nullptr},
    {"set_error", py_set_error, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) {
  const char* names[5] = {"data", "row_off", "scale", "zero", "col_scale"};
  for (int i = 0; i < 5; ++i)
    if (!(g_key[i] = PyUnicode_InternFromString(names[i]))) return nullptr;
  MatrixType.tp_name = "cobalt_amd._native.Matrix";
  MatrixType.tp_basicsize = sizeof(Matrix);
  MatrixType.tp_dealloc = matrix_dealloc;
  MatrixType.tp_flags = Py_TPFLAGS_DEFAULT;
  MatrixType.tp_new = matrix_new;
  if (PyType_Ready(&MatrixType) < 0) return nullptr;
  PyObject* m = PyModule_Create(&module_def);
  if (!m) return nullptr;
  g_error = PyExc_RuntimeError;
  Py_INCREF(g_error);
  Py_INCREF(&MatrixType);
  if (PyModule_AddObject(m, "Matrix", (PyObject*)&MatrixType) < 0) return nullptr;
  return m;
}
