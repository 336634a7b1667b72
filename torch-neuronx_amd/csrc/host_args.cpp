// Host side of a call, natively: allocates a call's outputs with the layout rules of the operator contract
// and writes its parameter block (include/mi355_sdpa.h).  A call whose kernels take a few microseconds is
// bound by the host that issues it, and two thirds of that time went into this work when it was done in
// Python: reading four shapes and strides per tensor, packing them, one torch.empty per output (forward:
// 10.7 of 14.7 us beside the 4 us launch; backward: 18 of 30 beside three).  Nothing here launches or decides anything:
// the block goes to the library's entry points as before, and so does every rule about layouts
// (mi355_sdpa_out_strides).
//
// A Python extension module on torch's own C++ tensors; the functions take positional arguments only.
#include <Python.h>

#include <ATen/Functions.h>
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
    const at::Tensor q = unit_last(query, hold), k = unit_last(key, hold), v = unit_last(value, hold);
    const int64_t B = q.size(0), H = q.size(1), L = q.size(2);
    out = like(query, {B, H, L, v.size(3)}, seq_major);
    if (need_lse) lse = at::empty({B, H, L}, query.options().dtype(at::kFloat));
    put(p->q, q), put(p->k, k), put(p->v, v), put(p->out, out, true), put(p->bias, bias);
  }
  p->lse = lse.defined() ? (float*)lse.mutable_data_ptr() : nullptr;
  p->bias_dtype = bias.defined() ? dtype_id(bias.scalar_type()) : 0;
  p->dtype = dtype_id(query.scalar_type());
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
  at::Tensor lse = tensor(a[6]);
  const bool is_causal = truth(a[9]), seq_major = truth(a[12]);
  const float scale = real(a[10]);
  const int32_t force_kernel = whole(a[11]);
  on_gpu(grad_out, "grad_out"), on_gpu(query, "query"), on_gpu(key, "key"), on_gpu(value, "value");
  std::vector<at::Tensor> hold;
  at::Tensor dq, dk, dv;
  {
    const Unlocked unlocked;
    const at::Tensor go = unit_last(grad_out, hold), q = unit_last(query, hold), k = unit_last(key, hold), v = unit_last(value, hold),
                     o = unit_last(out, hold);
    if (lse.scalar_type() != at::kFloat || !lse.is_contiguous()) hold.push_back(lse = lse.to(at::kFloat).contiguous());
    const int64_t B = q.size(0), Hq = q.size(1), L = q.size(2), E = q.size(3), Hkv = k.size(1), S = k.size(2), Dv = v.size(3);
    dq = like(query, {B, Hq, L, E}, seq_major), dk = like(key, {B, Hkv, S, E}, seq_major), dv = like(value, {B, Hkv, S, Dv}, seq_major);
    put(p->grad_out, go), put(p->q, q), put(p->k, k), put(p->v, v), put(p->out, o);
    put(p->grad_q, dq, true), put(p->grad_k, dk, true), put(p->grad_v, dv, true), put(p->bias, bias), put(p->grad_bias, dbias, true);
  }
  p->lse = (const float*)lse.const_data_ptr();
  p->bias_dtype = bias.defined() ? dtype_id(bias.scalar_type()) : 0;
  p->dtype = dtype_id(query.scalar_type());
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

// validate(q, k, v, has_bias, dropout_p, is_causal): the operator boundary's checks (mi355_sdpa_validate),
// RuntimeError with its message
PyObject* validate(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  arity(n, 6, "validate");
  const at::Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]);
  mi355_sdpa_desc d = {};
  auto fill = [](const at::Tensor& t, int32_t& dim, int64_t (&size)[4], int32_t& dtype, int32_t& last) {
    dim = (int32_t)t.dim(), dtype = dtype_id(t.scalar_type()), last = dim ? (int32_t)t.strides()[dim - 1] : 1;
    for (int i = 0; i < std::min<int>(4, dim); ++i) size[i] = t.sizes()[i];
  };
  fill(q, d.q_dim, d.q_size, d.q_dtype, d.q_last_stride);
  fill(k, d.k_dim, d.k_size, d.k_dtype, d.k_last_stride);
  fill(v, d.v_dim, d.v_size, d.v_dtype, d.v_last_stride);
  d.on_device = q.is_cuda() && k.is_cuda() && v.is_cuda();
  d.has_attn_bias = truth(a[3]), d.dropout_p = real(a[4]), d.is_causal = truth(a[5]);
  char msg[512];
  if (mi355_sdpa_validate(&d, msg, sizeof(msg)) != MI355_SDPA_OK) return PyErr_SetString(PyExc_RuntimeError, msg), nullptr;
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"validate", (PyCFunction)(void*)validate, METH_FASTCALL, "checks of the operator boundary"},
    {"forward", (PyCFunction)(void*)forward, METH_FASTCALL, "outputs and parameter block of a forward call"},
    {"backward", (PyCFunction)(void*)backward, METH_FASTCALL, "gradients and parameter block of a backward call"},
    {"decode", (PyCFunction)(void*)decode, METH_FASTCALL, "outputs and parameter block of an fp8 decode call"},
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
