// Host side of a call, natively: allocates a call's outputs with the layout rules of the operator contract
// and writes its parameter block (include/mi355_sdpa.h).  A call whose kernels take a few microseconds is
// bound by the host that issues it, and two thirds of that time went into this work when it was done in
// Python: reading four shapes and strides per tensor, packing them, one torch.empty per output (forward:
// 10.7 of 14.7 us beside the 4 us launch; backward: 18 of 30 beside three).  Nothing in this part launches or decides
// anything: the block goes to the library's entry points as before, and so does every rule about layouts
// (mi355_sdpa_out_strides).  The second part, "operators", serves the plain calls of torch's attention operators whole.
//
// A Python extension module on torch's own C++ tensors; the functions take positional arguments only.
#include <Python.h>

#include <ATen/Functions.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/InferenceMode.h>
#include <c10/hip/HIPStream.h>
#include <c10/util/Exception.h>
#include <torch/library.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/mi355_sdpa.h"

namespace {

int dtype_id(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return MI355_SDPA_F32;
    case at::kHalf: return MI355_SDPA_F16;
    case at::kBFloat16: return MI355_SDPA_BF16;
    case at::kDouble: return MI355_SDPA_F64;
    case at::kBool: return MI355_SDPA_BOOL;
    case at::kFloat8_e4m3fn: return MI355_SDPA_FP8_E4M3;
    default: return MI355_SDPA_OTHER;
  }
}

const at::Tensor& tensor(PyObject* o) {
  TORCH_CHECK_TYPE(THPVariable_Check(o), "expected a tensor, got ", Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}
// the caller's parameter block (never written through before it is known to be one)
template <typename P>
P* block(PyObject* o) {
  void* const p = PyLong_AsVoidPtr(o);
  if (PyErr_Occurred()) throw python_error();
  TORCH_CHECK_VALUE(p, "null parameter block");
  return (P*)p;
}
float real(PyObject* o) {
  const double x = PyFloat_AsDouble(o);
  if (PyErr_Occurred()) throw python_error();
  return (float)x;
}
int32_t whole(PyObject* o) {  // (whatever int() takes)
  PyObject* const i = PyNumber_Long(o);
  if (!i) throw python_error();
  const long x = PyLong_AsLong(i);
  Py_DECREF(i);
  if (PyErr_Occurred()) throw python_error();
  return (int32_t)x;
}
bool truth(PyObject* o) {
  const int x = PyObject_IsTrue(o);
  if (x < 0) throw python_error();
  return x;
}
// Other Python threads run while this lives: what allocates or copies may wait for the GPU (an allocator short of
// memory does).  The caller's tensors are held by value then, whatever those threads do to their Python objects.
struct Unlocked {
  PyThreadState* const state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};
at::Tensor optional(PyObject* o) { return o == Py_None ? at::Tensor() : tensor(o); }

void on_gpu(const at::Tensor& t, const char* name) {
  TORCH_CHECK_VALUE(t.is_cuda(), "Expected a GPU tensor for ", name, ", got ", t.device().str());
}
void four_dims(const at::Tensor& t) { TORCH_CHECK_VALUE(t.dim() == 4, "expected a 4-D tensor"); }

// unit stride on the head dim, as the kernels read rows; a copy is kept alive by the caller (`hold`)
at::Tensor unit_last(const at::Tensor& t, std::vector<at::Tensor>& hold) {
  four_dims(t);
  if (t.stride(3) == 1 || t.size(3) <= 1) return t;
  hold.push_back(t.contiguous());
  return hold.back();
}

// (written: a tensor that the call writes, whose memory must be nobody else's, a lazy clone's for instance)
void put(mi355_sdpa_tensor& d, const at::Tensor& t, bool written = false) {
  if (!t.defined()) return;
  four_dims(t);
  d.data = written ? t.mutable_data_ptr() : const_cast<void*>(t.const_data_ptr());
  for (int i = 0; i < 4; ++i) d.size[i] = t.sizes()[i], d.stride[i] = t.strides()[i];
}

using Shape = std::array<int64_t, 4>;

// New tensor of `shape` in the dimension order of `ref` (stride-0 dims never alias), with unit stride on
// the head dim; seq_major: laid out (B, L, H, D) in memory whatever `ref` is.
at::Tensor like(const at::Tensor& ref, const Shape& shape, bool seq_major) {
  if (seq_major) return at::empty({shape[0], shape[2], shape[1], shape[3]}, ref.options()).transpose(1, 2);
  if (ref.is_contiguous() && ref.numel() != 0) return at::empty(shape, ref.options());  // the common case needs no stride arithmetic
  int64_t st[4];
  mi355_sdpa_out_strides(ref.sizes().data(), ref.strides().data(), shape.data(), st);
  if (st[3] != 1 && shape[3] > 1) return at::empty(shape, ref.options());
  return at::empty_strided(shape, at::IntArrayRef(st, 4), ref.options());
}

PyObject* result(std::initializer_list<at::Tensor> outs, std::vector<at::Tensor>& hold) {
  PyObject* r = PyTuple_New((Py_ssize_t)outs.size() + 1);
  if (!r) return nullptr;
  Py_ssize_t i = 0;
  for (const at::Tensor& t : outs) PyTuple_SET_ITEM(r, i++, t.defined() ? THPVariable_Wrap(t) : (Py_INCREF(Py_None), Py_None));
  PyObject* h = PyTuple_New((Py_ssize_t)hold.size());
  if (!h) return Py_DECREF(r), nullptr;
  for (size_t j = 0; j < hold.size(); ++j) PyTuple_SET_ITEM(h, (Py_ssize_t)j, THPVariable_Wrap(hold[j]));
  PyTuple_SET_ITEM(r, i, h);
  return r;
}

void arity(Py_ssize_t got, Py_ssize_t want, const char* name) {
  TORCH_CHECK_TYPE(got == want, name, " takes ", want, " arguments, got ", got);
}

// outputs of a forward call, and its tensors in the block
void write_forward(mi355_sdpa_fwd_params& p, const at::Tensor& query, const at::Tensor& key, const at::Tensor& value, const at::Tensor& bias,
                   bool need_lse, bool seq_major, at::Tensor& out, at::Tensor& lse, std::vector<at::Tensor>& hold) {
  const at::Tensor q = unit_last(query, hold), k = unit_last(key, hold), v = unit_last(value, hold);
  const int64_t B = q.size(0), H = q.size(1), L = q.size(2);
  out = like(query, {B, H, L, v.size(3)}, seq_major);
  if (need_lse) lse = at::empty({B, H, L}, query.options().dtype(at::kFloat));
  put(p.q, q), put(p.k, k), put(p.v, v), put(p.out, out, true), put(p.bias, bias);
  p.lse = lse.defined() ? (float*)lse.mutable_data_ptr() : nullptr;
  p.bias_dtype = bias.defined() ? dtype_id(bias.scalar_type()) : 0;
  p.dtype = dtype_id(query.scalar_type());
}

// gradients of a backward call, and its tensors in the block
void write_backward(mi355_sdpa_bwd_params& p, const at::Tensor& grad_out, const at::Tensor& query, const at::Tensor& key, const at::Tensor& value,
                    const at::Tensor& out, at::Tensor lse, const at::Tensor& bias, const at::Tensor& dbias, bool seq_major, at::Tensor& dq,
                    at::Tensor& dk, at::Tensor& dv, std::vector<at::Tensor>& hold) {
  const at::Tensor go = unit_last(grad_out, hold), q = unit_last(query, hold), k = unit_last(key, hold), v = unit_last(value, hold),
                   o = unit_last(out, hold);
  if (lse.scalar_type() != at::kFloat || !lse.is_contiguous()) hold.push_back(lse = lse.to(at::kFloat).contiguous());
  const int64_t B = q.size(0), Hq = q.size(1), L = q.size(2), E = q.size(3), Hkv = k.size(1), S = k.size(2), Dv = v.size(3);
  dq = like(query, {B, Hq, L, E}, seq_major), dk = like(key, {B, Hkv, S, E}, seq_major), dv = like(value, {B, Hkv, S, Dv}, seq_major);
  put(p.grad_out, go), put(p.q, q), put(p.k, k), put(p.v, v), put(p.out, o);
  put(p.grad_q, dq, true), put(p.grad_k, dk, true), put(p.grad_v, dv, true), put(p.bias, bias), put(p.grad_bias, dbias, true);
  p.lse = (const float*)lse.const_data_ptr();
  p.bias_dtype = bias.defined() ? dtype_id(bias.scalar_type()) : 0;
  p.dtype = dtype_id(query.scalar_type());
}

// forward(block, q, k, v, bias, need_lse, is_causal, scale, force_kernel, seq_major) -> (out, lse or None, hold)
PyObject* forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 10, "forward");
  auto* p = block<mi355_sdpa_fwd_params>(a[0]);
  const at::Tensor query = tensor(a[1]), key = tensor(a[2]), value = tensor(a[3]), bias = optional(a[4]);
  const bool need_lse = truth(a[5]), is_causal = truth(a[6]), seq_major = truth(a[9]);
  const float scale = real(a[7]);
  const int32_t force_kernel = whole(a[8]);
  on_gpu(query, "query"), on_gpu(key, "key"), on_gpu(value, "value");
  std::vector<at::Tensor> hold;
  at::Tensor out, lse;
  {
    const Unlocked unlocked;
    write_forward(*p, query, key, value, bias, need_lse, seq_major, out, lse, hold);
  }
  p->is_causal = is_causal, p->scale = scale, p->force_kernel = force_kernel;
  return result({out, lse}, hold);
  END_HANDLE_TH_ERRORS
}

// backward(block, grad_out, q, k, v, out, lse, bias, grad_bias, is_causal, scale, force_kernel, seq_major)
//   -> (dq, dk, dv, hold)
PyObject* backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 13, "backward");
  auto* p = block<mi355_sdpa_bwd_params>(a[0]);
  const at::Tensor grad_out = tensor(a[1]), query = tensor(a[2]), key = tensor(a[3]), value = tensor(a[4]), out = tensor(a[5]),
                   bias = optional(a[7]), dbias = optional(a[8]);
  const at::Tensor lse = tensor(a[6]);
  const bool is_causal = truth(a[9]), seq_major = truth(a[12]);
  const float scale = real(a[10]);
  const int32_t force_kernel = whole(a[11]);
  on_gpu(grad_out, "grad_out"), on_gpu(query, "query"), on_gpu(key, "key"), on_gpu(value, "value");
  std::vector<at::Tensor> hold;
  at::Tensor dq, dk, dv;
  {
    const Unlocked unlocked;
    write_backward(*p, grad_out, query, key, value, out, lse, bias, dbias, seq_major, dq, dk, dv, hold);
  }
  p->is_causal = is_causal, p->scale = scale, p->force_kernel = force_kernel;
  return result({dq, dk, dv}, hold);
  END_HANDLE_TH_ERRORS
}

// decode(block, q, k, v, k_scale, v_scale, kv_lens, out, lse, need_lse, scale, num_splits) -> (out, lse or None, hold)
PyObject* decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 12, "decode");
  auto* p = block<mi355_sdpa_decode_params>(a[0]);
  const at::Tensor query = tensor(a[1]), key = tensor(a[2]), value = tensor(a[3]);
  const at::Tensor k_scale = optional(a[4]), v_scale = optional(a[5]), kv_lens = optional(a[6]);
  at::Tensor out = optional(a[7]), lse = optional(a[8]);
  const bool need_lse = truth(a[9]);
  const float scale = real(a[10]);
  const int32_t num_splits = whole(a[11]);
  on_gpu(query, "query"), on_gpu(key, "key"), on_gpu(value, "value");
  std::vector<at::Tensor> hold;
  {
    const Unlocked unlocked;
    const at::Tensor q = unit_last(query, hold), k = unit_last(key, hold), v = unit_last(value, hold);
    auto vec = [&](at::Tensor t, at::ScalarType dt) -> const void* {  // contiguous, on the query's device
      if (!t.defined()) return nullptr;
      if (t.scalar_type() != dt || !t.is_contiguous() || t.device() != query.device()) hold.push_back(t = t.to(query.device(), dt).contiguous());
      return t.const_data_ptr();
    };
    const int64_t B = q.size(0), H = q.size(1), L = q.size(2), D = v.size(3);
    if (!out.defined()) out = at::empty({B, H, L, D}, query.options());
    if (!lse.defined() && need_lse) lse = at::empty({B, H, L}, query.options().dtype(at::kFloat));
    TORCH_CHECK_VALUE(out.sizes() == at::IntArrayRef({B, H, L, D}) && out.scalar_type() == query.scalar_type(),
                      "decode_fp8kv: out must have shape (B, Hq, Lq, D) and the query's dtype");
    TORCH_CHECK_VALUE(!lse.defined() || (lse.sizes() == at::IntArrayRef({B, H, L}) && lse.scalar_type() == at::kFloat && lse.is_contiguous()),
                      "decode_fp8kv: lse must be a contiguous float32 (B, Hq, Lq) tensor");
    put(p->q, q), put(p->k, k), put(p->v, v), put(p->out, out, true);
    p->k_scale = (const float*)vec(k_scale, at::kFloat), p->v_scale = (const float*)vec(v_scale, at::kFloat);
    p->kv_lens = (const int32_t*)vec(kv_lens, at::kInt);
  }
  p->lse = lse.defined() ? (float*)lse.mutable_data_ptr() : nullptr;
  p->q_dtype = dtype_id(query.scalar_type());
  p->scale = scale, p->num_splits = num_splits;
  return result({out, lse}, hold);
  END_HANDLE_TH_ERRORS
}

mi355_sdpa_desc describe(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v) {
  mi355_sdpa_desc d = {};
  auto fill = [](const at::Tensor& t, int32_t& dim, int64_t (&size)[4], int32_t& dtype, int32_t& last) {
    dim = (int32_t)t.dim(), dtype = dtype_id(t.scalar_type()), last = dim ? (int32_t)t.strides()[dim - 1] : 1;
    for (int i = 0; i < std::min<int>(4, dim); ++i) size[i] = t.sizes()[i];
  };
  fill(q, d.q_dim, d.q_size, d.q_dtype, d.q_last_stride);
  fill(k, d.k_dim, d.k_size, d.k_dtype, d.k_last_stride);
  fill(v, d.v_dim, d.v_size, d.v_dtype, d.v_last_stride);
  d.on_device = q.is_cuda() && k.is_cuda() && v.is_cuda();
  return d;
}

// validate(q, k, v, has_bias, dropout_p, is_causal): the operator boundary's checks (mi355_sdpa_validate),
// RuntimeError with its message
PyObject* validate(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 6, "validate");
  mi355_sdpa_desc d = describe(tensor(a[0]), tensor(a[1]), tensor(a[2]));
  d.has_attn_bias = truth(a[3]), d.dropout_p = real(a[4]), d.is_causal = truth(a[5]);
  char msg[512];
  if (mi355_sdpa_validate(&d, msg, sizeof(msg)) != MI355_SDPA_OK) return PyErr_SetString(PyExc_RuntimeError, msg), nullptr;
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// ---- operators -------------------------------------------------------------------------------------------
// The flash and memory-efficient operators that F.scaled_dot_product_attention and its autograd formulas call, and their
// backwards.  A plain call (no bias, no dropout, float32 / float16 / bfloat16) is served here from the dispatcher to the
// launch; any other, and any that a check refuses, is the Python implementation's, which knows the rest of the rules and
// raises what it raised.  Through Python a forward takes 15 us of host time and a forward + backward 124, of which the
// kernels of a small layer are 25; here they take 7.5 and 49 (36 are what autograd takes around one product).  Beyond the
// boxing of arguments and results, each tensor that a graph saved went back through the interpreter when the graph was
// freed, in the autograd thread, against the main one.  What is left of the interpreter in a plain call is bound_kernel: its
// lock, two dictionary lookups and one small function, in a backward in the autograd thread.

struct Gil {
  const PyGILState_STATE state = PyGILState_Ensure();
  ~Gil() { PyGILState_Release(state); }
};
// An error of the interpreter, for code that runs without its lock (call with the lock held).
[[noreturn]] void raise() {
  python_error e;
  e.persist();
  throw e;
}

enum Op { kFlash, kFlashBackward, kEfficient, kEfficientBackward, kOps };
const char* const op_names[kOps] = {"_scaled_dot_product_flash_attention", "_scaled_dot_product_flash_attention_backward",
                                    "_scaled_dot_product_efficient_attention", "_scaled_dot_product_efficient_attention_backward"};
struct Operators {
  std::unique_ptr<torch::Library> library;
  PyObject* python[kOps];               // the Python implementations
  PyObject *ops, *impl;                 // namespaces of the modules `ops` and of the implementations
  PyObject *sdpa_forward, *sdpa_backward;  // ... and ops' own functions
  at::Tensor seed, offset;              // what a call without dropout returns for them (never written)
};
// (never destroyed: an operator may run as long as the process does)
Operators* operators = nullptr;

// The kernel that a call is bound to (TORCH_NEURONX_AMD_ENABLE_MFMA_SDPA, read on every call), or -1 where the Python
// implementation is to run: a program that has put its own function in the place of `ops.sdpa_forward` or
// `ops.sdpa_backward` sees the operators' calls.
int bound_kernel(bool backward) {
  const Gil gil;
  const char* const name = backward ? "sdpa_backward" : "sdpa_forward";
  if (PyDict_GetItemString(operators->ops, name) != (backward ? operators->sdpa_backward : operators->sdpa_forward)) return -1;
  PyObject* const f = PyDict_GetItemString(operators->impl, "_force_kernel");
  if (!f) return -1;
  PyObject* const r = PyObject_CallNoArgs(f);
  if (!r) raise();
  const long kernel = PyLong_AsLong(r);
  Py_DECREF(r);
  if (PyErr_Occurred()) raise();
  return (int)kernel;
}

bool plain(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, double dropout_p, bool is_causal) {
  if (dropout_p != 0. || !q.is_cuda() || k.device() != q.device() || v.device() != q.device() || q.dim() != 4 || q.size(3) == 0) return false;
  if (q.scalar_type() != at::kFloat && q.scalar_type() != at::kHalf && q.scalar_type() != at::kBFloat16) return false;
  mi355_sdpa_desc d = describe(q, k, v);
  d.is_causal = is_causal;
  return mi355_sdpa_validate(&d, nullptr, 0) == MI355_SDPA_OK;
}

float scale_of(const std::optional<double>& scale, const at::Tensor& q) { return (float)(scale ? *scale : 1. / std::sqrt((double)q.size(3))); }
void* stream_of(const at::Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
at::Tensor bytes_like(const at::Tensor& t, size_t n) { return at::empty({(int64_t)n}, t.options().dtype(at::kByte)); }

// (false: the Python implementation is to serve the call)
bool run_forward(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, double dropout_p, bool is_causal,
                 const std::optional<double>& scale, bool seq_major, at::Tensor& out, at::Tensor& lse) {
  if (!plain(q, k, v, dropout_p, is_causal)) return false;
  const int kernel = bound_kernel(false);
  if (kernel < 0) return false;
  const c10::DeviceGuard device(q.device());
  std::vector<at::Tensor> hold;
  mi355_sdpa_fwd_params p = {};
  write_forward(p, q, k, v, {}, true, seq_major, out, lse, hold);
  p.is_causal = is_causal, p.scale = scale_of(scale, q), p.force_kernel = kernel;
  if (q.size(2) <= 128) {  // few query rows: the library may want to split the keys over more workgroups
    if (const size_t need = mi355_sdpa_fwd_workspace_bytes(&p)) {
      hold.push_back(bytes_like(q, need));
      p.workspace = hold.back().mutable_data_ptr(), p.workspace_bytes = need;
    }
  }
  const int rc = mi355_sdpa_fwd(&p, stream_of(q));
  TORCH_CHECK(rc != MI355_SDPA_ERR_LAUNCH, mi355_sdpa_last_error());
  return rc == MI355_SDPA_OK;
}

bool run_backward(const at::Tensor& grad_out, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& out,
                  const at::Tensor& lse, double dropout_p, bool is_causal, const std::optional<double>& scale, bool seq_major, at::Tensor& dq,
                  at::Tensor& dk, at::Tensor& dv) {
  if (!plain(q, k, v, dropout_p, is_causal) || grad_out.scalar_type() != q.scalar_type() || grad_out.device() != q.device() ||
      out.device() != q.device() || lse.device() != q.device() || grad_out.dim() != 4 || out.dim() != 4)
    return false;
  const int kernel = bound_kernel(true);
  if (kernel < 0) return false;
  const c10::DeviceGuard device(q.device());
  std::vector<at::Tensor> hold;
  mi355_sdpa_bwd_params p = {};
  write_backward(p, grad_out, q, k, v, out, lse, {}, {}, seq_major, dq, dk, dv, hold);
  p.is_causal = is_causal, p.scale = scale_of(scale, q), p.force_kernel = kernel;
  const size_t need = mi355_sdpa_bwd_workspace_bytes(&p);
  hold.push_back(bytes_like(q, std::max<size_t>(need, 1)));
  p.workspace = hold.back().mutable_data_ptr(), p.workspace_bytes = need;
  const int rc = mi355_sdpa_bwd(&p, stream_of(q));
  TORCH_CHECK(rc != MI355_SDPA_ERR_LAUNCH, mi355_sdpa_last_error());
  return rc == MI355_SDPA_OK;
}

// The Python implementation of an operator: arguments in order, and the entries of the tuple it returns.
PyObject* wrap(const at::Tensor& t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}
PyObject* wrap(const std::optional<at::Tensor>& t) { return wrap(t ? *t : at::Tensor()); }
PyObject* wrap(double x) { return PyFloat_FromDouble(x); }
PyObject* wrap(bool x) { return PyBool_FromLong(x); }
PyObject* wrap(const c10::SymInt& x) { return PyLong_FromLongLong(x.expect_int()); }
PyObject* wrap(const std::optional<double>& x) {
  if (!x) Py_RETURN_NONE;
  return wrap(*x);
}
PyObject* wrap(const std::array<bool, 4>& x) {
  PyObject* const l = PyList_New(4);
  for (int i = 0; l && i < 4; ++i) PyList_SET_ITEM(l, i, wrap(bool(x[i])));
  return l;
}
template <size_t N, typename... A>
std::array<at::Tensor, N> python(Op op, const A&... args) {
  const Gil gil;
  PyObject* const in = PyTuple_New(sizeof...(A));
  if (!in) raise();
  Py_ssize_t i = 0;
  auto add = [&](PyObject* o) {
    if (!o) Py_DECREF(in), raise();
    PyTuple_SET_ITEM(in, i++, o);
  };
  (add(wrap(args)), ...);
  PyObject* const r = PyObject_CallObject(operators->python[op], in);
  Py_DECREF(in);
  if (!r) raise();
  std::array<at::Tensor, N> t;
  const bool whole = PyTuple_Check(r) && PyTuple_GET_SIZE(r) == (Py_ssize_t)N;
  for (size_t j = 0; whole && j < N; ++j)
    if (PyObject* const o = PyTuple_GET_ITEM(r, j); THPVariable_Check(o)) t[j] = THPVariable_Unpack(o);  // (None, a length: no tensor)
  Py_DECREF(r);
  TORCH_CHECK(whole, op_names[op], ": expected a tuple of ", N);
  return t;
}

using FlashOut = std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor, c10::SymInt, c10::SymInt, at::Tensor, at::Tensor, at::Tensor>;
FlashOut flash(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, double dropout_p, bool is_causal, bool debug_mask,
               std::optional<double> scale) {
  at::Tensor out, lse;
  if (!debug_mask && run_forward(q, k, v, dropout_p, is_causal, scale, false, out, lse))
    return {out, lse, at::Tensor(), at::Tensor(), q.size(2), k.size(2), operators->seed, operators->offset, at::empty({0}, q.options())};
  const auto r = python<9>(kFlash, q, k, v, dropout_p, is_causal, debug_mask, scale);
  return {r[0], r[1], r[2], r[3], q.size(2), k.size(2), r[6], r[7], r[8]};
}

std::tuple<at::Tensor, at::Tensor, at::Tensor> flash_backward(const at::Tensor& grad_out, const at::Tensor& q, const at::Tensor& k,
                                                              const at::Tensor& v, const at::Tensor& out, const at::Tensor& lse,
                                                              const at::Tensor& cum_q, const at::Tensor& cum_k, c10::SymInt max_q, c10::SymInt max_k,
                                                              double dropout_p, bool is_causal, const at::Tensor& seed, const at::Tensor& offset,
                                                              std::optional<double> scale) {
  at::Tensor dq, dk, dv;
  if (run_backward(grad_out, q, k, v, out, lse, dropout_p, is_causal, scale, false, dq, dk, dv)) return {dq, dk, dv};
  const auto r = python<3>(kFlashBackward, grad_out, q, k, v, out, lse, cum_q, cum_k, max_q, max_k, dropout_p, is_causal, seed, offset, scale);
  return {r[0], r[1], r[2]};
}

// (an empty bias is a lowering placeholder and counts as absent)
bool absent(const at::Tensor& bias) { return !bias.defined() || bias.numel() == 0; }

std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> efficient(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                                                                     const std::optional<at::Tensor>& bias, bool need_lse, double dropout_p,
                                                                     bool is_causal, std::optional<double> scale) {
  at::Tensor out, lse;
  if ((!bias || absent(*bias)) && run_forward(q, k, v, dropout_p, is_causal, scale, true, out, lse)) {
    if (!need_lse) lse = at::empty({q.size(0), q.size(1), 0}, lse.options());
    return {out, lse, operators->seed, operators->offset};
  }
  const auto r = python<4>(kEfficient, q, k, v, bias, need_lse, dropout_p, is_causal, scale);
  return {r[0], r[1], r[2], r[3]};
}

std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> efficient_backward(const at::Tensor& grad_out, const at::Tensor& q, const at::Tensor& k,
                                                                              const at::Tensor& v, const at::Tensor& bias, const at::Tensor& out,
                                                                              const at::Tensor& lse, const at::Tensor& seed, const at::Tensor& offset,
                                                                              double dropout_p, std::array<bool, 4> wanted, bool is_causal,
                                                                              std::optional<double> scale) {
  at::Tensor dq, dk, dv;
  if (absent(bias) && run_backward(grad_out, q, k, v, out, lse, dropout_p, is_causal, scale, true, dq, dk, dv))
    return {dq, dk, dv, at::empty({0}, q.options())};
  const auto r = python<4>(kEfficientBackward, grad_out, q, k, v, bias, out, lse, seed, offset, dropout_p, wanted, is_causal, scale);
  return {r[0], r[1], r[2], r[3]};
}

// register_operators(ops namespace, implementations' namespace): the four operators, for the dispatch key of the GPU.
PyObject* register_operators(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 2, "register_operators");
  TORCH_CHECK_TYPE(PyDict_Check(a[0]) && PyDict_Check(a[1]), "expected two namespaces");
  TORCH_CHECK_VALUE(!operators || !operators->library, "the operators are registered");
  auto get = [](PyObject* d, const char* name) {
    PyObject* const o = PyDict_GetItemString(d, name);
    TORCH_CHECK_VALUE(o, "no function ", name);
    Py_INCREF(o);
    return o;
  };
  if (!operators) {
    auto o = std::make_unique<Operators>();
    Py_INCREF(a[0]), Py_INCREF(a[1]);
    o->ops = a[0], o->impl = a[1];
    o->sdpa_forward = get(a[0], "sdpa_forward"), o->sdpa_backward = get(a[0], "sdpa_backward");
    for (int i = 0; i < kOps; ++i) o->python[i] = get(a[1], op_names[i] + 1);  // (the same name, without the underscore)
    const c10::InferenceMode normal(false);  // (an inference tensor could not be saved for a later backward)
    o->seed = at::zeros({}, at::kLong), o->offset = at::zeros({}, at::kLong);
    operators = o.release();
  }
  auto lib = std::make_unique<torch::Library>(torch::Library::IMPL, "aten", c10::DispatchKey::CUDA, __FILE__, __LINE__);
  struct Quiet : c10::WarningHandler {  // ("overriding a previously registered kernel" is the point)
    void process(const c10::Warning&) override {}
  } quiet;
  const c10::WarningUtils::WarningHandlerGuard guard(&quiet);
  lib->impl(op_names[kFlash], flash);
  lib->impl(op_names[kFlashBackward], flash_backward);
  lib->impl(op_names[kEfficient], efficient);
  lib->impl(op_names[kEfficientBackward], efficient_backward);
  operators->library = std::move(lib);
  PyObject* const names = PyTuple_New(kOps);
  for (int i = 0; names && i < kOps; ++i) PyTuple_SET_ITEM(names, i, PyUnicode_FromString(op_names[i]));
  return names;
  END_HANDLE_TH_ERRORS
}

// unregister_operators(): the stock kernels come back
PyObject* unregister_operators(PyObject*, PyObject* const*, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 0, "unregister_operators");
  if (operators) operators->library.reset();
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"validate", (PyCFunction)(void*)validate, METH_FASTCALL, "checks of the operator boundary"},
    {"forward", (PyCFunction)(void*)forward, METH_FASTCALL, "outputs and parameter block of a forward call"},
    {"backward", (PyCFunction)(void*)backward, METH_FASTCALL, "gradients and parameter block of a backward call"},
    {"decode", (PyCFunction)(void*)decode, METH_FASTCALL, "outputs and parameter block of an fp8 decode call"},
    {"register_operators", (PyCFunction)(void*)register_operators, METH_FASTCALL, "torch's attention operators, served here"},
    {"unregister_operators", (PyCFunction)(void*)unregister_operators, METH_FASTCALL, "... and no longer"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_args", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host_args(void) {
  PyObject* m = PyModule_Create(&module);
  // (the binding checks these against its own structures)
  if (m && (PyModule_AddIntConstant(m, "FWD_BYTES", sizeof(mi355_sdpa_fwd_params)) || PyModule_AddIntConstant(m, "BWD_BYTES", sizeof(mi355_sdpa_bwd_params)) ||
            PyModule_AddIntConstant(m, "DECODE_BYTES", sizeof(mi355_sdpa_decode_params))))
    return Py_DECREF(m), nullptr;
  return m;
}
