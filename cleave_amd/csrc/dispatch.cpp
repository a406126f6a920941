// The host side of a compiled kernel's call, in one native step: check the tensors against the kernel's
// declared parameters, work out the run-time extents, allocate the outputs and the scratch, fill in the
// argument arrays and hand the launches to libcleave_hip.so on the caller's current stream.
//
// In Python the same steps (parsing the grid expressions, ctypes descriptors, one torch allocation per
// split partial, a device context) took 37 us per kernel and twice that for a split pair: more than any
// kernel of the small operators.  Here a call costs what its allocations and launches cost.
//
// A call that does not match (wrong type, rank, extent, layout or device, a subclass that is not a
// tensor, an extent that makes the grid too large) returns NotImplemented and nothing has happened: the
// Python path then takes the call and names what is wrong.
//
// No state is kept from call to call, so any number of threads and streams may share a plan: scratch is
// allocated per call from torch's allocator on the current stream and given back at the end of it (the
// allocator hands it out again in stream order only).
#include <Python.h>

#include <ATen/Context.h>
#include <ATen/EmptyTensor.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/record_function.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <cstdlib>
#include <string>
#include <vector>

namespace {

typedef int (*launch_fn)(void* fn, const uint32_t grid[3], const uint32_t block[3], uint32_t lds, void* stream,
                         void** args, int nargs);

// ---- extents: integers, or expressions over the run-time dims in postfix form ----------------------
enum Op : int64_t { CONST_, DIM, ADD, SUB, MUL, FLOORDIV, MOD, NEG, CEILDIV, MIN_, MAX_ };
typedef std::vector<int64_t> Expr;

int64_t floor_div(int64_t a, int64_t b) {
  const int64_t q = a / b;
  return (a % b != 0 && ((a < 0) != (b < 0))) ? q - 1 : q;
}

// false: a division by zero, or a dim that is not known
bool evaluate(const Expr& e, const int64_t* dims, int64_t* out) {
  int64_t st[32];
  int n = 0;
  for (size_t i = 0; i < e.size(); ++i) {
    switch (e[i]) {
      case CONST_: st[n++] = e[++i]; continue;
      case DIM: st[n] = dims[e[++i]]; if (st[n] < 0) return false; ++n; continue;
      case NEG: st[n - 1] = -st[n - 1]; continue;
      default: break;
    }
    const int64_t b = st[--n], a = st[n - 1];
    int64_t r = 0;
    switch (e[i]) {
      case ADD: r = a + b; break;
      case SUB: r = a - b; break;
      case MUL: r = a * b; break;
      case MIN_: r = a < b ? a : b; break;
      case MAX_: r = a > b ? a : b; break;
      default:
        if (b == 0) return false;
        r = e[i] == FLOORDIV ? floor_div(a, b) : e[i] == MOD ? a - floor_div(a, b) * b : -floor_div(-a, b);
    }
    st[n - 1] = r;
  }
  *out = st[0];
  return n == 1;
}

// postfix programs come from Python already checked for operand counts; the depth is checked here
bool read_expr(PyObject* o, Expr* e) {
  PyObject* seq = PySequence_Fast(o, "an extent is a sequence of integers");
  if (!seq) return false;
  int depth = 0;
  bool ok = true;
  for (Py_ssize_t i = 0; ok && i < PySequence_Fast_GET_SIZE(seq); ++i) {
    const int64_t v = PyLong_AsLongLong(PySequence_Fast_GET_ITEM(seq, i));
    if (v == -1 && PyErr_Occurred()) { Py_DECREF(seq); return false; }
    e->push_back(v);
    if (v == CONST_ || v == DIM) {
      if (++i >= PySequence_Fast_GET_SIZE(seq)) { ok = false; break; }
      e->push_back(PyLong_AsLongLong(PySequence_Fast_GET_ITEM(seq, i)));
      if (++depth > 32) ok = false;
    } else if (v == NEG) {
      if (depth < 1) ok = false;
    } else {
      if (--depth < 1 || v < 0 || v > MAX_) ok = false;
    }
  }
  Py_DECREF(seq);
  if (!ok || depth != 1) { PyErr_SetString(PyExc_ValueError, "malformed extent program"); return false; }
  return !PyErr_Occurred();
}

enum ArgKind { TENSOR, F32, I32 };
struct Arg {
  int kind;
  at::ScalarType dtype;
  uintptr_t misaligned;          // TENSOR: address bits that have to be zero (the kernel's loads need them so)
  std::vector<int64_t> dim;      // TENSOR, per axis: >= 0 an extent; -1 - d binds run-time dim d; INT64_MIN an expression
  std::vector<Expr> expr;        // the expressions, in axis order
};
struct Out {
  at::ScalarType dtype;
  std::vector<Expr> shape;
};
enum ValueKind { V_ARG, V_OUT, V_TEMP, V_DIM };
struct Value { int kind, index; };
struct Launch {
  void* fn;
  Expr grid[3];
  uint32_t block[3], lds;
  bool optional;                 // left out where its grid is empty; any other empty grid means that the call has nothing to do
  std::vector<Value> values;
};

struct Plan {
  PyObject_HEAD
  vectorcallfunc vectorcall;
  std::vector<Arg>* args;
  std::vector<Expr>* derived;
  std::vector<Out>* outs;
  std::vector<Expr>* temps;      // bytes of each scratch buffer
  std::vector<Launch>* launches;
  int n_dims;                    // bound by the arguments; the derived ones follow
  int result;                    // 0: None, 1: a tensor or a list of tensors, 2: a tensor or a tuple
  PyObject* keep;                // what the function handles belong to
  PyObject* raw_stream;          // device index -> the current stream's handle
  PyObject* fail;                // status of a launch that failed -> raises
  launch_fn launch;
};

constexpr int kMaxDims = 32, kMaxValues = 64, kMaxOuts = 8, kMaxTemps = 16;

at::ScalarType scalar_type(const char* name) {
  const std::string s(name);
  if (s == "float16") return at::kHalf;
  if (s == "bfloat16") return at::kBFloat16;
  if (s == "float32") return at::kFloat;
  if (s == "int32") return at::kInt;
  return at::ScalarType::Undefined;
}

#define MISS() do { Py_RETURN_NOTIMPLEMENTED; } while (0)

// A tensor whose sizes and memory are what they seem: not fake or traced (Python key), batched or wrapped by a
// transform (vmap, grad), a zero without memory, or a lazy negation.  The others go through torch's own accessors in
// the Python path, which raise what they always raised.
bool plain(const at::Tensor& t) {
  constexpr c10::DispatchKeySet others({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::FuncTorchBatched,
                                        c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize, c10::DispatchKey::ZeroTensor,
                                        c10::DispatchKey::Negative, c10::DispatchKey::Conjugate});
  return t.defined() && !t.key_set().has_any(others) && t.has_storage();
}

// Whether an allocation may go to torch's allocator without passing its dispatcher: nobody listens there -- no mode, transform
// or tracer on this thread, no profiler -- and fresh memory needs no fill.  A call of a paged decode operator (two outputs)
// takes 5.6 us of host time instead of 6.2 with this and its split / single rule in plain integers, a small matmul 4.0 instead of
// 4.2; both are what such calls are bound by.
bool dispatcher_idle() {
  const auto included = c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set;
  return included.empty() && !at::hasCallbacks() &&
         !(at::globalContext().deterministicAlgorithms() && at::globalContext().deterministicFillUninitializedMemory());
}

// The allocator behind torch's device tensors, one for the life of the process: asked of a tensor, because the one registered
// for the device type makes storage of the type's HIP twin.
c10::Allocator* device_allocator(int device) {
  static c10::Allocator* const its = at::empty({1}, at::TensorOptions().device(at::kCUDA, device).dtype(at::kByte)).storage().allocator();
  return its;
}

PyObject* call_plain(PyObject* self_, PyObject* const* argv, size_t nargsf, PyObject* kwnames) {
  Plan* self = reinterpret_cast<Plan*>(self_);
  const size_t n = PyVectorcall_NARGS(nargsf);
  const std::vector<Arg>& spec = *self->args;
  if (n != spec.size() || (kwnames && PyTuple_GET_SIZE(kwnames))) MISS();
  if (getenv("CLEAVE_POISON_BUFFERS")) MISS();          // (the Python path fills fresh buffers with NaN)

  int64_t dims[kMaxDims];
  for (int i = 0; i < kMaxDims; ++i) dims[i] = -1;
  union Slot { void* p; float f; int32_t i; };
  Slot arg_value[kMaxValues];
  int device = -1;
  bool deferred = false;
  for (size_t i = 0; i < n; ++i) {
    const Arg& a = spec[i];
    PyObject* o = argv[i];
    if (a.kind != TENSOR) {
      double v;
      if (PyFloat_CheckExact(o)) v = PyFloat_AS_DOUBLE(o);
      else if (PyLong_CheckExact(o)) { v = PyLong_AsDouble(o); if (v == -1.0 && PyErr_Occurred()) { PyErr_Clear(); MISS(); } }
      else MISS();
      if (a.kind == F32) arg_value[i].f = (float)v;
      else { if (v != (double)(int32_t)v) MISS(); arg_value[i].i = (int32_t)v; }
      continue;
    }
    if (!THPVariable_Check(o)) MISS();
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!plain(t)) MISS();
    if (t.layout() != at::kStrided || t.device().type() != at::kCUDA || t.scalar_type() != a.dtype || !t.is_contiguous()) MISS();
    if (device < 0) device = t.device().index();
    else if (device != t.device().index()) MISS();
    const auto sizes = t.sizes();
    if (sizes.size() != a.dim.size()) MISS();
    for (size_t k = 0; k < sizes.size(); ++k) {
      const int64_t want = a.dim[k];
      if (want >= 0) { if (sizes[k] != want) MISS(); }
      else if (want == INT64_MIN) deferred = true;
      else {
        int64_t& d = dims[-1 - want];
        if (d < 0) d = sizes[k];
        else if (d != sizes[k]) MISS();
      }
    }
    arg_value[i].p = t.mutable_data_ptr();
    if (reinterpret_cast<uintptr_t>(arg_value[i].p) & a.misaligned) MISS();
  }
  if (device < 0) MISS();
  for (int i = 0; i < self->n_dims; ++i) if (dims[i] < 0) MISS();
  if (deferred) {
    for (size_t i = 0; i < n; ++i) {
      const Arg& a = spec[i];
      if (a.kind != TENSOR || a.expr.empty()) continue;
      const auto sizes = THPVariable_Unpack(argv[i]).sizes();
      size_t e = 0;
      for (size_t k = 0; k < a.dim.size(); ++k) {
        if (a.dim[k] != INT64_MIN) continue;
        int64_t v;
        if (!evaluate(a.expr[e++], dims, &v) || v != sizes[k]) MISS();
      }
    }
  }
  for (size_t i = 0; i < self->derived->size(); ++i) {
    int64_t v;
    if (!evaluate((*self->derived)[i], dims, &v) || v < 0) MISS();
    dims[self->n_dims + i] = v;
  }
  int32_t dim_value[kMaxDims];
  for (int i = 0; i < kMaxDims; ++i) {
    if (dims[i] > INT32_MAX) MISS();
    dim_value[i] = (int32_t)dims[i];
  }
  uint32_t grids[8][3];
  bool empty = false, left_out[8] = {};
  for (size_t l = 0; l < self->launches->size(); ++l)
    for (int k = 0; k < 3; ++k) {
      int64_t v;
      if (!evaluate((*self->launches)[l].grid[k], dims, &v)) MISS();
      if (v < 1) ((*self->launches)[l].optional ? left_out[l] : empty) = true;
      else if (v > (k == 0 ? (int64_t)INT32_MAX : 65535)) MISS();
      else grids[l][k] = (uint32_t)v;
    }

  if (c10::impl::VirtualGuardImpl(c10::DeviceType::CUDA).getDevice().index() != device) MISS();
  const auto on_device = at::TensorOptions().device(at::kCUDA, device);
  const bool direct = dispatcher_idle() && device_allocator(device);
  c10::Allocator* const allocator = direct ? device_allocator(device) : nullptr;
  constexpr c10::DispatchKeySet cuda_keys(c10::DispatchKey::CUDA);
  auto fresh = [&](at::IntArrayRef shape, at::ScalarType dtype) -> at::Tensor {
    if (!direct) return at::empty(shape, on_device.dtype(dtype));
    return at::Tensor(at::detail::empty_generic(shape, allocator, cuda_keys, dtype, std::nullopt));
  };
  at::Tensor outs[kMaxOuts];
  void* out_ptr[kMaxOuts];
  for (size_t i = 0; i < self->outs->size(); ++i) {
    const Out& o = (*self->outs)[i];
    int64_t shape[8];
    for (size_t k = 0; k < o.shape.size(); ++k)
      if (!evaluate(o.shape[k], dims, &shape[k]) || shape[k] < 0) MISS();
    outs[i] = fresh(at::IntArrayRef(shape, o.shape.size()), o.dtype);
    out_ptr[i] = outs[i].data_ptr();
  }
  at::Tensor scratch;
  void* temp_ptr[kMaxTemps];
  if (!self->temps->empty() && !empty) {
    int64_t at_byte[kMaxTemps], total = 0;
    for (size_t i = 0; i < self->temps->size(); ++i) {
      int64_t v;
      if (!evaluate((*self->temps)[i], dims, &v) || v < 0) MISS();
      at_byte[i] = total;
      total += (v + 255) / 256 * 256;
    }
    // (nothing where only launches that are left out have scratch)
    if (total) scratch = fresh({total}, at::kByte);
    char* const base = total ? static_cast<char*>(scratch.data_ptr()) : nullptr;
    for (size_t i = 0; i < self->temps->size(); ++i) temp_ptr[i] = base + at_byte[i];
  }
  if (!empty) {
    PyObject* index = PyLong_FromLong(device);
    if (!index) return nullptr;
    PyObject* handle = PyObject_CallOneArg(self->raw_stream, index);
    Py_DECREF(index);
    if (!handle) return nullptr;
    void* stream = PyLong_AsVoidPtr(handle);
    Py_DECREF(handle);
    if (PyErr_Occurred()) return nullptr;
    // (a launch waits where the stream's queue is full: other threads run meanwhile)
    PyThreadState* released = PyEval_SaveThread();
    int failed = 0;
    for (size_t l = 0; l < self->launches->size() && !failed; ++l) {
      const Launch& q = (*self->launches)[l];
      if (left_out[l]) continue;
      void* values[kMaxValues];
      int nv = 0;
      for (const Value& v : q.values)
        values[nv++] = v.kind == V_ARG ? (void*)&arg_value[v.index] : v.kind == V_OUT ? (void*)&out_ptr[v.index]
                       : v.kind == V_TEMP ? (void*)&temp_ptr[v.index] : (void*)&dim_value[v.index];
      failed = self->launch(q.fn, grids[l], q.block, q.lds, stream, values, nv);
    }
    PyEval_RestoreThread(released);
    if (failed) {
      // (the error types of the library's Python binding; its error text is this thread's own)
      PyObject* none = PyObject_CallFunction(self->fail, "i", failed);
      Py_XDECREF(none);
      if (!PyErr_Occurred()) PyErr_Format(PyExc_RuntimeError, "a launch failed with status %d", failed);
      return nullptr;
    }
  }
  if (self->result == 0) Py_RETURN_NONE;
  const size_t n_out = self->outs->size();
  if (n_out == 1) return THPVariable_Wrap(std::move(outs[0]));
  PyObject* many = self->result == 1 ? PyList_New(n_out) : PyTuple_New(n_out);
  if (!many) return nullptr;
  for (size_t i = 0; i < n_out; ++i) {
    PyObject* t = THPVariable_Wrap(std::move(outs[i]));
    if (!t) { Py_DECREF(many); return nullptr; }
    if (self->result == 1) PyList_SET_ITEM(many, i, t);
    else PyTuple_SET_ITEM(many, i, t);
  }
  return many;
}

// (no C++ exception may leave a C entry)
PyObject* call(PyObject* self, PyObject* const* argv, size_t nargsf, PyObject* kwnames) {
  try {
    return call_plain(self, argv, nargsf, kwnames);
  } catch (const std::exception& e) {
    // an allocation that failed, say: torch's own error type is raised by the Python path's allocation
    PyErr_Clear();
    MISS();
  }
}

// ---- construction ----------------------------------------------------------------------------------
bool bad(const char* what) { PyErr_SetString(PyExc_ValueError, what); return false; }

template <class F>
bool for_each(PyObject* o, F f) {
  PyObject* seq = PySequence_Fast(o, "expected a sequence");
  if (!seq) return false;
  bool ok = true;
  for (Py_ssize_t i = 0; ok && i < PySequence_Fast_GET_SIZE(seq); ++i) ok = f(PySequence_Fast_GET_ITEM(seq, i));
  Py_DECREF(seq);
  return ok;
}

bool read_plan(Plan* p, PyObject* args, PyObject* derived, PyObject* outs, PyObject* temps, PyObject* launches) {
  if (!for_each(args, [&](PyObject* o) {
        Arg a;
        const char* dtype;
        PyObject* dims;
        unsigned align;
        if (!PyArg_ParseTuple(o, "isOI", &a.kind, &dtype, &dims, &align)) return false;
        if (align == 0 || (align & (align - 1))) return bad("an alignment is a power of two");
        a.misaligned = align - 1;
        a.dtype = scalar_type(dtype);
        if (a.kind == TENSOR && a.dtype == at::ScalarType::Undefined) return bad("unknown element type");
        if (!for_each(dims, [&](PyObject* d) {
              if (PyLong_Check(d)) {
                const int64_t v = PyLong_AsLongLong(d);
                if (v < -(int64_t)p->n_dims) return bad("a dim beyond the declared ones");
                a.dim.push_back(v);
                return !PyErr_Occurred();
              }
              Expr e;
              if (!read_expr(d, &e)) return false;
              a.dim.push_back(INT64_MIN);
              a.expr.push_back(e);
              return true;
            }))
          return false;
        p->args->push_back(a);
        return true;
      }))
    return false;
  if (!for_each(derived, [&](PyObject* o) { Expr e; if (!read_expr(o, &e)) return false; p->derived->push_back(e); return true; })) return false;
  if (!for_each(outs, [&](PyObject* o) {
        Out out;
        const char* dtype;
        PyObject* shape;
        if (!PyArg_ParseTuple(o, "sO", &dtype, &shape)) return false;
        out.dtype = scalar_type(dtype);
        if (out.dtype == at::ScalarType::Undefined) return bad("unknown element type");
        if (!for_each(shape, [&](PyObject* d) { Expr e; if (!read_expr(d, &e)) return false; out.shape.push_back(e); return true; })) return false;
        if (out.shape.size() > 8) return bad("an output of more than eight axes");
        p->outs->push_back(out);
        return true;
      }))
    return false;
  if (!for_each(temps, [&](PyObject* o) { Expr e; if (!read_expr(o, &e)) return false; p->temps->push_back(e); return true; })) return false;
  if (!for_each(launches, [&](PyObject* o) {
        Launch l;
        unsigned long long fn;
        PyObject *grid, *values;
        unsigned bx, by, bz, lds;
        int optional = 0;
        if (!PyArg_ParseTuple(o, "KO(III)IO|i", &fn, &grid, &bx, &by, &bz, &lds, &values, &optional)) return false;
        l.optional = optional != 0;
        l.fn = reinterpret_cast<void*>(fn);
        l.block[0] = bx; l.block[1] = by; l.block[2] = bz;
        l.lds = lds;
        int k = 0;
        if (!for_each(grid, [&](PyObject* d) { return k < 3 ? read_expr(d, &l.grid[k++]) : bad("a grid of more than three extents"); })) return false;
        if (k != 3) return bad("a grid of three extents");
        if (!for_each(values, [&](PyObject* d) {
              Value v;
              if (!PyArg_ParseTuple(d, "ii", &v.kind, &v.index)) return false;
              const int limit[4] = {(int)p->args->size(), (int)p->outs->size(), (int)p->temps->size(), p->n_dims + (int)p->derived->size()};
              if (v.kind < 0 || v.kind > V_DIM || v.index < 0 || v.index >= limit[v.kind]) return bad("a launch argument that names nothing");
              l.values.push_back(v);
              return true;
            }))
          return false;
        if (l.values.size() > kMaxValues) return bad("too many launch arguments");
        p->launches->push_back(l);
        return true;
      }))
    return false;
  if (p->args->size() > kMaxValues || p->n_dims + (int)p->derived->size() > kMaxDims || p->outs->size() > kMaxOuts ||
      p->temps->size() > kMaxTemps || p->launches->size() > 8 || p->launches->empty())
    return bad("a plan beyond the dispatcher's limits");
  // every dim that an expression names exists
  const int known = p->n_dims + (int)p->derived->size();
  auto inside = [&](const Expr& e) {
    for (size_t i = 0; i < e.size(); ++i)
      if (e[i] == CONST_) ++i;
      else if (e[i] == DIM && (e[++i] < 0 || e[i] >= known)) return false;
    return true;
  };
  bool ok = true;
  for (auto& a : *p->args) for (auto& e : a.expr) ok = ok && inside(e);
  for (auto& e : *p->derived) ok = ok && inside(e);
  for (auto& o : *p->outs) for (auto& e : o.shape) ok = ok && inside(e);
  for (auto& e : *p->temps) ok = ok && inside(e);
  for (auto& l : *p->launches) for (auto& e : l.grid) ok = ok && inside(e);
  return ok || bad("an extent names an unknown dim");
}

void plan_dealloc(PyObject* o) {
  Plan* p = reinterpret_cast<Plan*>(o);
  delete p->args; delete p->derived; delete p->outs; delete p->temps; delete p->launches;
  Py_XDECREF(p->keep);
  Py_XDECREF(p->raw_stream);
  Py_XDECREF(p->fail);
  Py_TYPE(o)->tp_free(o);
}

PyTypeObject PlanType = {PyVarObject_HEAD_INIT(nullptr, 0) "cleave_amd._dispatch.Plan"};

// make_plan(args, n_dims, derived, outs, temps, launches, result, keep, raw_stream, fail, launch address)
PyObject* make_plan(PyObject*, PyObject* a) {
  PyObject *args, *derived, *outs, *temps, *launches, *keep, *raw, *fail;
  int n_dims, result;
  unsigned long long launch;
  if (!PyArg_ParseTuple(a, "OiOOOOiOOOK", &args, &n_dims, &derived, &outs, &temps, &launches, &result, &keep, &raw, &fail, &launch)) return nullptr;
  Plan* p = PyObject_New(Plan, &PlanType);
  if (!p) return nullptr;
  p->vectorcall = call;
  p->args = new std::vector<Arg>; p->derived = new std::vector<Expr>; p->outs = new std::vector<Out>;
  p->temps = new std::vector<Expr>; p->launches = new std::vector<Launch>;
  p->n_dims = n_dims;
  p->result = result;
  Py_INCREF(keep); p->keep = keep;
  Py_INCREF(raw); p->raw_stream = raw;
  Py_INCREF(fail); p->fail = fail;
  p->launch = reinterpret_cast<launch_fn>(launch);
  if (!read_plan(p, args, derived, outs, temps, launches)) { Py_DECREF(p); return nullptr; }
  return reinterpret_cast<PyObject*>(p);
}

PyMethodDef methods[] = {{"make_plan", make_plan, METH_VARARGS, "a callable that checks, allocates and launches"}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_dispatch", "native calls of compiled kernels", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__dispatch() {
  PlanType.tp_basicsize = sizeof(Plan);
  PlanType.tp_dealloc = plan_dealloc;
  PlanType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
  PlanType.tp_vectorcall_offset = offsetof(Plan, vectorcall);
  PlanType.tp_call = PyVectorcall_Call;
  PlanType.tp_doc = "One compiled operator's call";
  if (PyType_Ready(&PlanType) < 0) return nullptr;
  return PyModule_Create(&module_def);
}
