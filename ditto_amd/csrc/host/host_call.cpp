// The call path from torch tensors to the C ABI of the chain library, in native code: a descriptor is filled from the
// tensors' shapes, strides and types, checked, and handed over with the data pointers and torch's current stream.
//
// What it is for: the smallest chains run for two or three microseconds beside a launch, and the same work done tensor
// attribute by tensor attribute in Python took 7 - 9 us per call (22 us for an attention module's call, five view
// operations included), so the host and not the device set the pace.
//
// A Python extension module (ditto_amd/_host.so) over torch's C++ interface; it holds no state of its own beyond the
// objects Python creates from its two types.
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Exceptions.h>
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <cstring>
#include <string>
#include <vector>

#include "../../../include/ditto_chain.h"

namespace {

// ---- small helpers ---------------------------------------------------------------------------
struct PyFail {};  // a Python exception is set

[[noreturn]] void fail(PyObject* type, const std::string& what) {
  PyErr_SetString(type, what.c_str());
  throw PyFail();
}

const at::Tensor& tensor_of(PyObject* o) {
  if (!THPVariable_Check(o)) fail(PyExc_TypeError, std::string("expected a torch tensor, got ") + Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kHalf: return DITTO_F16;
    case at::kBFloat16: return DITTO_BF16;
    case at::kFloat: return DITTO_F32;
    case at::kDouble: return DITTO_F64;
    case at::kChar: return DITTO_I8;
    case at::kInt: return DITTO_I32;
    default: fail(PyExc_ValueError, std::string("unsupported tensor dtype ") + c10::toString(t));
  }
}

std::string shape_text(at::IntArrayRef s) {
  std::string r = "(";
  for (size_t i = 0; i < s.size(); ++i) r += (i ? ", " : "") + std::to_string(s[i]);
  return r + (s.size() == 1 ? ",)" : ")");
}

int inter_code(PyObject* o) {
  if (PyUnicode_Check(o)) {
    static const struct { const char* name; int code; } names[] = {{"cast", DITTO_INTER_CAST}, {"relu", DITTO_INTER_RELU},
                                                                   {"softmax", DITTO_INTER_SOFTMAX}, {"requant", DITTO_INTER_REQUANT}};
    for (const auto& n : names)
      if (PyUnicode_CompareWithASCIIString(o, n.name) == 0) return n.code;
    PyErr_SetObject(PyExc_KeyError, o);
    throw PyFail();
  }
  const long v = PyLong_AsLong(o);
  if (v == -1 && PyErr_Occurred()) throw PyFail();
  return (int)v;
}

double number(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw PyFail();
  return v;
}
long integer(PyObject* o) {
  const long v = PyLong_AsLong(o);
  if (v == -1 && PyErr_Occurred()) throw PyFail();
  return v;
}
bool truth(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw PyFail();
  return v != 0;
}

template <typename F>
PyObject* guarded(F&& f) {
  try {
    return f();
  } catch (const PyFail&) {
    return nullptr;
  } catch (const c10::Error& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
    return nullptr;
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

void check_device(const at::Tensor* const* t, int n) {
  const c10::Device dev = t[0]->device();
  if (dev.type() != c10::kCUDA)
    fail(PyExc_ValueError, "fused chains run on a HIP device; got a " + c10::DeviceTypeName(dev.type(), true) + " tensor");
  for (int i = 1; i < n; ++i)
    if (t[i]->device() != dev) fail(PyExc_ValueError, "all tensors of a chain must be on the same device");
}

// `launch(stream)` on torch's current stream of the tensors' device, made current for the call, without the GIL
template <typename F>
int on_current_stream(const c10::Device& dev, F&& launch) {
  c10::OptionalDeviceGuard guard;
  if (c10::hip::current_device() != dev.index()) guard.reset_device(dev);
  void* const stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
  PyThreadState* const state = PyEval_SaveThread();
  const int rc = launch(stream);
  PyEval_RestoreThread(state);
  return rc;
}

// ---- batched matrix chains -------------------------------------------------------------------
// one operand as [outer][batch][rows][cols] with its strides
struct Operand {
  int64_t outer = 1, outer_stride = 0, batch, rows, cols, sb, sr, sc;
};

Operand operand_of(const at::Tensor& t, const char* name) {
  const auto s = t.sizes(), st = t.strides();
  Operand o;
  switch (t.dim()) {
    case 2: o.batch = 1, o.rows = s[0], o.cols = s[1], o.sb = s[0] * st[0], o.sr = st[0], o.sc = st[1]; break;
    case 3: o.batch = s[0], o.rows = s[1], o.cols = s[2], o.sb = st[0], o.sr = st[1], o.sc = st[2]; break;
    case 4:
      o.outer = s[0], o.outer_stride = st[0];
      o.batch = s[1], o.rows = s[2], o.cols = s[3], o.sb = st[1], o.sr = st[2], o.sc = st[3];
      break;
    default: fail(PyExc_ValueError, std::string(name) + " must be [batch, rows, cols] or [rows, cols]");
  }
  return o;
}

struct BmmParams {
  int inter;
  float softmax_scale, requant_scale;
  int tile_variant;
  bool relu_out;
};

std::string dims(std::initializer_list<int64_t> v, const char* last = nullptr) {
  std::string r = "[";
  bool first = true;
  for (int64_t x : v) r += (first ? "" : ", ") + std::to_string(x), first = false;
  return r + (last ? std::string(", ") + last : "") + "]";
}

void fill_bmm(ditto_bmm_chain_desc* d, const Operand& A, const Operand& B, const Operand& C, const Operand& F,
              at::ScalarType in, at::ScalarType out, const BmmParams& p) {
  memset(d, 0, sizeof(*d));
  d->abi_version = DITTO_CHAIN_ABI_VERSION;
  d->in_dtype = dtype_code(in);
  d->acc_dtype = in == at::kChar ? DITTO_I32 : in == at::kDouble ? DITTO_F64 : DITTO_F32;
  d->out_dtype = dtype_code(out);
  d->inter_op = p.inter;
  if (B.sc == 1 || B.cols == 1) {
    d->b_layout = DITTO_B_KL;
    d->b_row_stride = B.sr;
  } else if (B.sr == 1) {
    d->b_layout = DITTO_B_LK;
    d->b_row_stride = B.sc;
  } else {
    fail(PyExc_ValueError, "B must be contiguous along L or along K");
  }
  d->batch = A.batch * A.outer;
  d->M = A.rows, d->N = C.cols, d->K = A.cols, d->L = B.cols;
  d->batch_inner = A.outer > 1 ? A.batch : 0;
  d->a_batch_stride_outer = A.outer_stride, d->b_batch_stride_outer = B.outer_stride;
  d->c_batch_stride_outer = C.outer_stride, d->f_batch_stride_outer = F.outer_stride;
  d->a_batch_stride = A.sb, d->a_row_stride = A.sr;
  d->b_batch_stride = B.sb;
  d->c_batch_stride = C.sb, d->c_row_stride = C.sr;
  d->f_batch_stride = F.sb, d->f_row_stride = F.sr;
  d->softmax_scale = p.softmax_scale;
  d->requant_scale = p.requant_scale;
  d->tile_variant = p.tile_variant;
  d->relu_out = p.relu_out;
}

void fill_bmm(ditto_bmm_chain_desc* d, const at::Tensor& a, const at::Tensor& b, const at::Tensor& c, const at::Tensor& f,
              const BmmParams& p) {
  const Operand A = operand_of(a, "A"), B = operand_of(b, "B"), C = operand_of(c, "C"), F = operand_of(f, "F");
  if (A.outer != B.outer || A.outer != C.outer || A.outer != F.outer)
    fail(PyExc_ValueError, "A, B, C, F must agree in their outer batch extent");
  if (B.batch != A.batch || B.rows != A.cols)
    fail(PyExc_ValueError, "B must be [batch, K, L] = " + dims({A.batch, A.cols}, "L") + ", got " + shape_text({B.batch, B.rows, B.cols}));
  if (C.batch != A.batch || C.rows != B.cols)
    fail(PyExc_ValueError, "C must be [batch, L, N] = " + dims({A.batch, B.cols}, "N") + ", got " + shape_text({C.batch, C.rows, C.cols}));
  if (F.batch != A.batch || F.rows != A.rows || F.cols != C.cols)
    fail(PyExc_ValueError, "F must be " + dims({A.batch, A.rows, C.cols}) + ", got " + shape_text({F.batch, F.rows, F.cols}));
  if (a.scalar_type() != b.scalar_type() || a.scalar_type() != c.scalar_type())
    fail(PyExc_ValueError, "A, B, C must share one dtype");
  for (const auto& [o, name] : {std::pair<const Operand*, const char*>{&A, "A"}, {&C, "C"}, {&F, "F"}})
    if (o->cols > 1 && o->sc != 1) fail(PyExc_ValueError, std::string(name) + " rows must be contiguous");
  fill_bmm(d, A, B, C, F, a.scalar_type(), f.scalar_type(), p);
}

int run_bmm(const ditto_bmm_chain_desc& d, const at::Tensor& a, const at::Tensor& b, const at::Tensor& c, const at::Tensor& f,
            PyObject* aux_obj) {
  const void* aux = nullptr;
  if (aux_obj && aux_obj != Py_None) {
    const at::Tensor& x = tensor_of(aux_obj);
    const at::Tensor* both[2] = {&a, &x};
    check_device(both, 2);
    if (x.scalar_type() != at::kFloat || !x.is_contiguous() || x.numel() != d.L)
      fail(PyExc_ValueError, "aux must be a contiguous fp32 tensor of L = " + std::to_string(d.L) + " scales");
    aux = x.data_ptr();
  }
  const void *pa = a.data_ptr(), *pb = b.data_ptr(), *pc = c.data_ptr();
  void* const pf = f.data_ptr();
  return on_current_stream(a.device(), [&](void* stream) {
    return ditto_bmm_chain_run(&d, pa, pb, pc, aux, pf, nullptr, 0, stream);
  });
}

// fill_bmm_desc(address, A, B, C, F, inter_op, softmax_scale, requant_scale, tile_variant, relu_out)
PyObject* py_fill_bmm_desc(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 10) fail(PyExc_TypeError, "fill_bmm_desc takes 10 arguments");
    auto* d = static_cast<ditto_bmm_chain_desc*>(PyLong_AsVoidPtr(v[0]));
    if (!d) fail(PyExc_ValueError, "null descriptor");
    const BmmParams p = {inter_code(v[5]), (float)number(v[6]), (float)number(v[7]), (int)integer(v[8]), truth(v[9])};
    fill_bmm(d, tensor_of(v[1]), tensor_of(v[2]), tensor_of(v[3]), tensor_of(v[4]), p);
    Py_RETURN_NONE;
  });
}

// run_bmm(A, B, C, F, inter_op, softmax_scale, requant_scale, aux, tile_variant, relu_out) -> return code
PyObject* py_run_bmm(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 10) fail(PyExc_TypeError, "run_bmm takes 10 arguments");
    const at::Tensor &a = tensor_of(v[0]), &b = tensor_of(v[1]), &c = tensor_of(v[2]), &f = tensor_of(v[3]);
    const at::Tensor* all[4] = {&a, &b, &c, &f};
    check_device(all, 4);
    const BmmParams p = {inter_code(v[4]), (float)number(v[5]), (float)number(v[6]), (int)integer(v[8]), truth(v[9])};
    ditto_bmm_chain_desc d;
    fill_bmm(&d, a, b, c, f, p);
    return PyLong_FromLong(run_bmm(d, a, b, c, f, v[7]));
  });
}

// run_bmm_desc(address, A, B, C, F, aux) -> return code
PyObject* py_run_bmm_desc(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 6) fail(PyExc_TypeError, "run_bmm_desc takes 6 arguments");
    const auto* d = static_cast<const ditto_bmm_chain_desc*>(PyLong_AsVoidPtr(v[0]));
    if (!d) fail(PyExc_ValueError, "null descriptor");
    const at::Tensor &a = tensor_of(v[1]), &b = tensor_of(v[2]), &c = tensor_of(v[3]), &f = tensor_of(v[4]);
    const at::Tensor* all[4] = {&a, &b, &c, &f};
    check_device(all, 4);
    return PyLong_FromLong(run_bmm(*d, a, b, c, f, v[5]));
  });
}

// Attention over a packed projection x [batch, M, 3 * hidden] into out [batch, M, hidden]: the descriptor of the chain over
// [batch, heads, M, d] views of the packed rows (keys as stored, one row of d per key); false where the tensors are not the
// plain case (a 3-D projection with contiguous rows, a contiguous out).
bool plain_projection(const at::Tensor& x, int64_t heads, int64_t hidden) {
  return x.dim() == 3 && x.size(2) == 3 * hidden && x.stride(2) == 1 && x.device().type() == c10::kCUDA && x.size(0) > 0 &&
         x.size(1) > 0 && hidden / heads > 1;
}
bool plain_output(const at::Tensor& o, const at::Tensor& x, int64_t hidden) {
  return o.dim() == 3 && o.size(0) == x.size(0) && o.size(1) == x.size(1) && o.size(2) == hidden && o.is_contiguous() &&
         o.device() == x.device();
}
void fill_attention(ditto_bmm_chain_desc* desc, const at::Tensor& x, at::ScalarType out, int64_t heads, int64_t hidden, float scale,
                    int tile_variant) {
  const int64_t batch = x.size(0), M = x.size(1), d = hidden / heads, s0 = x.stride(0), s1 = x.stride(1);
  Operand Q, K, F;
  Q.outer = batch, Q.outer_stride = s0, Q.batch = heads, Q.rows = M, Q.cols = d, Q.sb = d, Q.sr = s1, Q.sc = 1;
  K = Q, K.rows = d, K.cols = M, K.sr = 1, K.sc = s1;
  F = Q, F.outer_stride = M * hidden, F.sr = hidden;
  fill_bmm(desc, Q, K, Q, F, x.scalar_type(), out, {DITTO_INTER_SOFTMAX, scale, 1.f, tile_variant, false});
}

// run_attention(query_key_value, out | None, heads, hidden, scale, tile_variant) -> (return code, out), or None where the
// tensors are not the plain case (then the caller goes by views)
PyObject* py_run_attention(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 6) fail(PyExc_TypeError, "run_attention takes 6 arguments");
    const at::Tensor& x = tensor_of(v[0]);
    const int64_t heads = integer(v[2]), hidden = integer(v[3]);
    if (!plain_projection(x, heads, hidden)) Py_RETURN_NONE;
    at::Tensor made;
    PyObject* out_obj = v[1];
    if (out_obj != Py_None) {
      if (!plain_output(tensor_of(out_obj), x, hidden)) Py_RETURN_NONE;
    } else {
      made = at::empty({x.size(0), x.size(1), hidden}, x.options().requires_grad(false));
    }
    const at::Tensor& out = out_obj != Py_None ? tensor_of(out_obj) : made;
    ditto_bmm_chain_desc desc;
    fill_attention(&desc, x, out.scalar_type(), heads, hidden, (float)number(v[4]), (int)integer(v[5]));
    const int64_t step = hidden * x.element_size();
    const char* const base = static_cast<const char*>(x.data_ptr());
    void* const dst = out.data_ptr();
    const int rc = on_current_stream(x.device(), [&](void* stream) {
      return ditto_bmm_chain_run(&desc, base, base + step, base + 2 * step, nullptr, dst, nullptr, 0, stream);
    });
    PyObject* result = PyTuple_New(2);
    if (!result) throw PyFail();
    PyTuple_SET_ITEM(result, 0, PyLong_FromLong(rc));
    if (out_obj != Py_None) {
      Py_INCREF(out_obj);
      PyTuple_SET_ITEM(result, 1, out_obj);
    } else {
      PyTuple_SET_ITEM(result, 1, THPVariable_Wrap(std::move(made)));
    }
    return result;
  });
}

// run_attention_sets(projections, outs, heads, hidden, scale, tile_variant, batch, rows): run_attention on several projections
// [batch, rows, 3 * hidden], in as few launches as hold them -> return code, or None where that does not do: tensors that are
// not the plain case, not of that shape or not alike, or an output that shares memory with another set's tensors (then the caller runs them in order)
// attention_sets_launches(the same): how many launches that call makes (or its return code where it fails), or None likewise
template <typename Call>
PyObject* attention_sets(PyObject* const* v, Py_ssize_t n, Call&& call) {
  return guarded([&]() -> PyObject* {
    if (n != 8 || !PyList_Check(v[0]) || !PyList_Check(v[1]) || PyList_GET_SIZE(v[0]) != PyList_GET_SIZE(v[1]) ||
        PyList_GET_SIZE(v[0]) == 0)
      fail(PyExc_TypeError, "attention sets take two lists of tensors, equally long, and 6 numbers");
    const int64_t heads = integer(v[2]), hidden = integer(v[3]);
    const Py_ssize_t sets = PyList_GET_SIZE(v[0]);
    struct Span {
      uintptr_t begin, end;
      bool meets(const Span& o) const { return begin < o.end && o.begin < end; }
    };
    std::vector<Span> in(sets), out(sets);
    std::vector<const void*> q(sets), k(sets), c(sets);
    std::vector<void*> f(sets);
    const int64_t batch = integer(v[6]), rows = integer(v[7]);
    const at::Tensor &x0 = tensor_of(PyList_GET_ITEM(v[0], 0)), &o0 = tensor_of(PyList_GET_ITEM(v[1], 0));
    const int64_t step = hidden * (int64_t)x0.element_size();
    for (Py_ssize_t i = 0; i < sets; ++i) {
      const at::Tensor &x = tensor_of(PyList_GET_ITEM(v[0], i)), &o = tensor_of(PyList_GET_ITEM(v[1], i));
      if (!plain_projection(x, heads, hidden) || !plain_output(o, x, hidden) || x.size(0) != batch || x.size(1) != rows ||
          x.strides() != x0.strides() || x.scalar_type() != x0.scalar_type() || o.scalar_type() != o0.scalar_type() ||
          x.device() != x0.device())
        Py_RETURN_NONE;
      const char* const base = static_cast<const char*>(x.data_ptr());
      q[i] = base, k[i] = base + step, c[i] = base + 2 * step, f[i] = o.data_ptr();
      const int64_t last = (x.size(0) - 1) * x.stride(0) + (x.size(1) - 1) * x.stride(1) + x.size(2);
      in[i] = {reinterpret_cast<uintptr_t>(base), reinterpret_cast<uintptr_t>(base) + last * x.element_size()};
      out[i] = {reinterpret_cast<uintptr_t>(f[i]), reinterpret_cast<uintptr_t>(f[i]) + o.numel() * o.element_size()};
    }
    for (Py_ssize_t i = 0; i < sets; ++i)
      for (Py_ssize_t j = 0; j < sets; ++j)
        if (i != j && (out[i].meets(in[j]) || out[i].meets(out[j]))) Py_RETURN_NONE;
    ditto_bmm_chain_desc desc;
    fill_attention(&desc, x0, o0.scalar_type(), heads, hidden, (float)number(v[4]), (int)integer(v[5]));
    return PyLong_FromLong(on_current_stream(x0.device(), [&](void* stream) {
      return call(&desc, (int)sets, q.data(), k.data(), c.data(), f.data(), stream);
    }));
  });
}
PyObject* py_run_attention_sets(PyObject*, PyObject* const* v, Py_ssize_t n) { return attention_sets(v, n, ditto_bmm_chain_run_sets); }
PyObject* py_attention_sets_launches(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return attention_sets(v, n, [](const ditto_bmm_chain_desc* d, int sets, const void* const* q, const void* const* k, const void* const* c,
                                 void* const* f, void*) { return ditto_bmm_chain_sets_launches(d, sets, q, k, c, f); });
}

// ---- a built function's call -----------------------------------------------------------------
// shapes of the arguments as the schedule declares them
struct Shapes {
  int count = 0;
  int dim[8];
  int64_t size[8][5];
  std::string name[8];
  void read(PyObject* seq) {  // a sequence of (name, shape)
    PyObject* const fast = PySequence_Fast(seq, "argument shapes must be a sequence");
    if (!fast) throw PyFail();
    count = (int)PySequence_Fast_GET_SIZE(fast);
    if (count > 8) fail(PyExc_ValueError, "too many arguments");
    for (int i = 0; i < count; ++i) {
      const char* nm;
      PyObject* shape;
      if (!PyArg_ParseTuple(PySequence_Fast_GET_ITEM(fast, i), "sO!", &nm, &PyTuple_Type, &shape)) throw PyFail();
      name[i] = nm;
      dim[i] = (int)PyTuple_GET_SIZE(shape);
      if (dim[i] > 5) fail(PyExc_ValueError, "too many dimensions");
      for (int k = 0; k < dim[i]; ++k) size[i][k] = integer(PyTuple_GET_ITEM(shape, k));
    }
    Py_DECREF(fast);
  }
  bool same(int i, const at::Tensor& t) const {
    if (t.dim() != dim[i]) return false;
    const auto s = t.sizes();
    for (int k = 0; k < dim[i]; ++k)
      if (s[k] != size[i][k]) return false;
    return true;
  }
  void check(int i, const at::Tensor& t) const {
    if (!same(i, t))
      fail(PyExc_ValueError, "argument for " + name[i] + " has shape " + shape_text(t.sizes()) + ", expected " +
                                 shape_text(at::IntArrayRef(size[i], dim[i])));
  }
};

// BmmCall(arguments, inter_op, softmax_scale, requant_scale, tile_variant, relu_out, has_scale): called with the tensors
// in schedule order (A, B, C[, scale], F), returns the library's return code
struct BmmCall {
  PyObject_HEAD
  Shapes* shapes;
  BmmParams params;
  bool has_scale;
};

int bmm_call_init(PyObject* self, PyObject* args, PyObject*) {
  auto* s = reinterpret_cast<BmmCall*>(self);
  PyObject *shapes, *inter;
  double sm, rq;
  int tile, relu, scale;
  if (!PyArg_ParseTuple(args, "OOddipp", &shapes, &inter, &sm, &rq, &tile, &relu, &scale)) return -1;
  PyObject* ok = guarded([&]() -> PyObject* {
    if (!s->shapes) s->shapes = new Shapes();
    s->shapes->read(shapes);
    s->params = {inter_code(inter), (float)sm, (float)rq, tile, relu != 0};
    s->has_scale = scale != 0;
    if (s->shapes->count != (s->has_scale ? 5 : 4)) fail(PyExc_ValueError, "a matrix chain takes A, B, C[, scale], F");
    Py_RETURN_NONE;
  });
  if (!ok) return -1;
  Py_DECREF(ok);
  return 0;
}
void bmm_call_free(PyObject* self) {
  delete reinterpret_cast<BmmCall*>(self)->shapes;
  Py_TYPE(self)->tp_free(self);
}
PyObject* bmm_call_call(PyObject* self, PyObject* args, PyObject*) {
  const auto* s = reinterpret_cast<const BmmCall*>(self);
  return guarded([&]() -> PyObject* {
    const Py_ssize_t n = PyTuple_GET_SIZE(args);
    if (!s->shapes || n != s->shapes->count)
      fail(PyExc_ValueError, "expected " + std::to_string(s->shapes ? s->shapes->count : 0) +
                                 " tensors (inputs then outputs), got " + std::to_string(n));
    for (int i = 0; i < n; ++i) s->shapes->check(i, tensor_of(PyTuple_GET_ITEM(args, i)));
    const at::Tensor &a = tensor_of(PyTuple_GET_ITEM(args, 0)), &b = tensor_of(PyTuple_GET_ITEM(args, 1)),
                     &c = tensor_of(PyTuple_GET_ITEM(args, 2)), &f = tensor_of(PyTuple_GET_ITEM(args, n - 1));
    ditto_bmm_chain_desc d;
    fill_bmm(&d, a, b, c, f, s->params);
    const at::Tensor* all[4] = {&a, &b, &c, &f};
    check_device(all, 4);
    return PyLong_FromLong(run_bmm(d, a, b, c, f, s->has_scale ? PyTuple_GET_ITEM(args, 3) : nullptr));
  });
}

// ConvCall(arguments): the repeated call of a built conv chain.  remember(address, X, Y, workspace | None, W1 | None,
// W2 | None) keeps the descriptor that fits tensors like X and Y, the workspace and, for a function whose workspace holds
// the repacked weights, the weight tensors it was made from.  A call with (X, W1, W2, Y) runs the chain and returns the
// library's return code if the tensors are like those remembered (and the weights the bound ones, unchanged), else None:
// everything else is the caller's.
struct ConvCall {
  PyObject_HEAD
  Shapes* shapes;
  ditto_conv_chain_desc desc;
  bool ready, bound;
  at::ScalarType in, out;
  c10::Device* device;
  at::Tensor *workspace, *w1, *w2;
  uint32_t v1, v2;
};

int conv_call_init(PyObject* self, PyObject* args, PyObject*) {
  auto* s = reinterpret_cast<ConvCall*>(self);
  PyObject* shapes;
  if (!PyArg_ParseTuple(args, "O", &shapes)) return -1;
  PyObject* ok = guarded([&]() -> PyObject* {
    if (!s->shapes) {
      s->shapes = new Shapes();
      s->device = new c10::Device(c10::kCPU);
      s->workspace = new at::Tensor(), s->w1 = new at::Tensor(), s->w2 = new at::Tensor();
    }
    s->ready = false;
    s->shapes->read(shapes);
    if (s->shapes->count != 4) fail(PyExc_ValueError, "a conv chain takes X, W1, W2, Y");
    Py_RETURN_NONE;
  });
  if (!ok) return -1;
  Py_DECREF(ok);
  return 0;
}
void conv_call_free(PyObject* self) {
  auto* s = reinterpret_cast<ConvCall*>(self);
  delete s->shapes;
  delete s->device;
  delete s->workspace;
  delete s->w1;
  delete s->w2;
  Py_TYPE(self)->tp_free(self);
}
uint32_t version_of(const at::Tensor& t) { return t.unsafeGetTensorImpl()->version_counter().current_version(); }

PyObject* conv_call_remember(PyObject* self, PyObject* const* v, Py_ssize_t n) {
  auto* s = reinterpret_cast<ConvCall*>(self);
  return guarded([&]() -> PyObject* {
    if (n != 6 || !s->shapes) fail(PyExc_TypeError, "remember takes 6 arguments");
    s->ready = false;
    const auto* d = static_cast<const ditto_conv_chain_desc*>(PyLong_AsVoidPtr(v[0]));
    if (!d) fail(PyExc_ValueError, "null descriptor");
    const at::Tensor &x = tensor_of(v[1]), &y = tensor_of(v[2]);
    s->desc = *d;
    s->in = x.scalar_type(), s->out = y.scalar_type();
    *s->device = x.device();
    *s->workspace = v[3] != Py_None ? tensor_of(v[3]) : at::Tensor();
    s->bound = v[4] != Py_None;
    *s->w1 = s->bound ? tensor_of(v[4]) : at::Tensor();
    *s->w2 = s->bound ? tensor_of(v[5]) : at::Tensor();
    // (tensors without a version counter cannot be told from updated ones)
    if (s->bound && (s->w1->is_inference() || s->w2->is_inference())) Py_RETURN_NONE;
    if (s->bound) s->v1 = version_of(*s->w1), s->v2 = version_of(*s->w2);
    s->ready = true;
    Py_RETURN_NONE;
  });
}
PyObject* conv_call_forget(PyObject* self, PyObject*) {
  reinterpret_cast<ConvCall*>(self)->ready = false;
  Py_RETURN_NONE;
}
PyObject* conv_call_call(PyObject* self, PyObject* args, PyObject*) {
  const auto* s = reinterpret_cast<const ConvCall*>(self);
  return guarded([&]() -> PyObject* {
    if (!s->ready || PyTuple_GET_SIZE(args) != 4) Py_RETURN_NONE;
    const at::Tensor* t[4];
    for (int i = 0; i < 4; ++i) {
      PyObject* const o = PyTuple_GET_ITEM(args, i);
      if (!THPVariable_Check(o)) Py_RETURN_NONE;
      t[i] = &THPVariable_Unpack(o);
      if (!s->shapes->same(i, *t[i]) || t[i]->scalar_type() != (i == 3 ? s->out : s->in) || t[i]->device() != *s->device ||
          !t[i]->is_contiguous())
        Py_RETURN_NONE;
    }
    if (s->bound) {
      // the bound tensor itself or another view of exactly its memory (views share the version counter)
      if (t[1]->is_inference() || t[2]->is_inference()) Py_RETURN_NONE;
      if (t[1]->data_ptr() != s->w1->data_ptr() || t[2]->data_ptr() != s->w2->data_ptr() || version_of(*t[1]) != s->v1 ||
          version_of(*t[2]) != s->v2)
        Py_RETURN_NONE;
    }
    void* const ws = s->workspace->defined() ? s->workspace->data_ptr() : nullptr;
    const size_t ws_bytes = ws ? (size_t)s->workspace->numel() * s->workspace->element_size() : 0;
    const void *x = t[0]->data_ptr(), *w1 = t[1]->data_ptr(), *w2 = t[2]->data_ptr();
    void* const y = t[3]->data_ptr();
    const bool bound = s->bound;
    const ditto_conv_chain_desc d = s->desc;
    return PyLong_FromLong(on_current_stream(*s->device, [&](void* stream) {
      return bound ? ditto_conv_chain_run_prepared(&d, x, w1, w2, y, ws, ws_bytes, stream)
                   : ditto_conv_chain_run(&d, x, w1, w2, y, ws, ws_bytes, stream);
    }));
  });
}

PyMethodDef conv_call_methods[] = {
    {"remember", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(conv_call_remember)), METH_FASTCALL, nullptr},
    {"forget", conv_call_forget, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyTypeObject bmm_call_type = {PyVarObject_HEAD_INIT(nullptr, 0)};
PyTypeObject conv_call_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

#define FAST(name, fn) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(fn)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST("fill_bmm_desc", py_fill_bmm_desc), FAST("run_bmm", py_run_bmm),
                         FAST("run_bmm_desc", py_run_bmm_desc), FAST("run_attention", py_run_attention),
                         FAST("run_attention_sets", py_run_attention_sets),
                         FAST("attention_sets_launches", py_attention_sets_launches),
                         {nullptr, nullptr, 0, nullptr}};
#undef FAST

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "native call path of the fused chains", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
  bmm_call_type.tp_name = "ditto_amd._host.BmmCall";
  bmm_call_type.tp_basicsize = sizeof(BmmCall);
  bmm_call_type.tp_flags = Py_TPFLAGS_DEFAULT;
  bmm_call_type.tp_new = PyType_GenericNew;
  bmm_call_type.tp_init = bmm_call_init;
  bmm_call_type.tp_dealloc = bmm_call_free;
  bmm_call_type.tp_call = bmm_call_call;
  conv_call_type.tp_name = "ditto_amd._host.ConvCall";
  conv_call_type.tp_basicsize = sizeof(ConvCall);
  conv_call_type.tp_flags = Py_TPFLAGS_DEFAULT;
  conv_call_type.tp_new = PyType_GenericNew;
  conv_call_type.tp_init = conv_call_init;
  conv_call_type.tp_dealloc = conv_call_free;
  conv_call_type.tp_call = conv_call_call;
  conv_call_type.tp_methods = conv_call_methods;
  if (PyType_Ready(&bmm_call_type) < 0 || PyType_Ready(&conv_call_type) < 0) return nullptr;
  PyObject* m = PyModule_Create(&module);
  if (!m) return nullptr;
  Py_INCREF(&bmm_call_type);
  Py_INCREF(&conv_call_type);
  if (PyModule_AddObject(m, "BmmCall", reinterpret_cast<PyObject*>(&bmm_call_type)) < 0 ||
      PyModule_AddObject(m, "ConvCall", reinterpret_cast<PyObject*>(&conv_call_type)) < 0)
    return nullptr;
  return m;
}
