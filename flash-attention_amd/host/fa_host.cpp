// The calls of flash_attn_gfx950.fwd / bwd (and their block-sparse forms), and of the passes around them, made natively: arguments checked, outputs and scratch
// allocated, the argument struct of the C ABI filled and the entry point called, without Python in between.
//
// Every check the Python binding makes is made here too, but nothing is reported: a call that fails one, or that is of a kind
// handled there (probabilities returned, profiling events, a device that is not current, tensors without memory of their own such as those of
// functorch and of fake-tensor tracing), returns None and the binding runs it - and raises what it has to.  What the library itself refuses
// is raised here with the binding's text.
//
// Bound by the interpreter.  us with the binding's own calls / with these: one forward of 12 heads x 61 tokens (kernel 6) 21.4 / 14.2; training
// steps of 8 x 12 x 256 .. 512 with dropout (kernels 56; an empty autograd function with a backward takes 48) 159 / 101, 8 x 12 x 1024 rotary
// (110) 175 / 118, 8 x 8 x 421 .. 701 with a bias (100) 208 / 149 - 100 where both host threads, the
// caller's and the autograd engine's, run on one core: handing over to another core is what the rest goes to.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/flash_attn_gfx950.h"

namespace {

struct Library {
  int (*fwd)(const fa_fwd_args*);
  int (*fwd_block)(const fa_fwd_args*);
  int (*bwd)(const fa_bwd_args*);
  int (*bwd_block)(const fa_bwd_args*);
  size_t (*fwd_workspace_bytes)(const fa_fwd_args*);
  size_t (*bwd_workspace_bytes)(const fa_bwd_args*);
  void (*round_seqlens)(int32_t, int32_t, int32_t, int32_t, int32_t*, int32_t*);
  const char* (*last_error)();
  int (*pad_bias_rows)(const void*, void*, int32_t, int32_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, void*);
  int (*bias_grad_reduce_ragged)(const void*, void*, const fa_bwd_args*, int32_t, int32_t, int64_t, int64_t, int64_t);
  int (*rotary)(const fa_rotary_args*);
  int (*token_positions)(const int32_t*, int32_t, int32_t, int32_t*, void*);
} g_lib;
bool g_bound = false;

// bind(addresses of the twelve entry points above, in their order)
PyObject* py_bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  constexpr int kEntries = 12;
  if (n != kEntries) return PyErr_Format(PyExc_TypeError, "bind takes %d addresses", kEntries);
  void* f[kEntries];
  for (int i = 0; i < kEntries; i++) {
    f[i] = PyLong_AsVoidPtr(a[i]);
    if (!f[i]) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null address");
      return nullptr;
    }
  }
  static_assert(sizeof(g_lib) == sizeof(f), "a pointer each");
  memcpy(&g_lib, f, sizeof(f));
  g_bound = true;
  Py_RETURN_NONE;
}

// A tensor argument; null for None.  ok is cleared for anything but a plain tensor (or parameter) with memory of its own.
const at::Tensor* tensor(PyObject* o, bool& ok) {
  if (o == Py_None) return nullptr;
  if (!THPVariable_Check(o)) {
    ok = false;
    return nullptr;
  }
  const at::Tensor& t = THPVariable_Unpack(o);
  constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::Functionalize, c10::DispatchKey::FuncTorchGradWrapper,
                                         c10::DispatchKey::FuncTorchBatched});
  if (!t.defined() || !t.has_storage() || t.key_set().has_any(wrapped) || t.layout() != at::kStrided) ok = false;
  return &t;
}
bool as_int(PyObject* o, int64_t* v) {  // a Python int (what int() of anything else gives is left to the binding)
  if (!PyLong_Check(o)) return false;
  int overflow = 0;
  *v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0 && !(*v == -1 && PyErr_Occurred()) && *v >= INT32_MIN && *v <= INT32_MAX;
}
bool as_double(PyObject* o, double* v) {
  if (PyFloat_Check(o)) *v = PyFloat_AS_DOUBLE(o);
  else if (PyLong_Check(o)) *v = PyLong_AsDouble(o);
  else return false;
  if (!PyErr_Occurred()) return true;
  PyErr_Clear();  // (an int beyond a double: the binding meets it again)
  return false;
}
bool as_flag(PyObject* o, int32_t* v) {
  const int r = PyObject_IsTrue(o);
  if (r < 0) PyErr_Clear();  // (something without a truth value, as above)
  *v = r > 0;
  return r >= 0;
}
inline void* ptr(const at::Tensor& t) { return t.data_ptr(); }

struct Shape {
  at::ScalarType dtype;
  c10::Device device{c10::kCPU};
  int64_t heads, dim, batch, total_q, total_k;
};
bool rows_ok(const at::Tensor* t, const Shape& s, int64_t total) {
  return t && t->is_cuda() && t->device() == s.device && t->scalar_type() == s.dtype && t->dim() == 3 && t->size(0) == total &&
         t->size(1) == s.heads && t->size(2) == s.dim && t->stride(2) == 1;
}
bool cu_ok(const at::Tensor* t, const Shape& s) {
  return t && t->is_cuda() && t->device() == s.device && t->scalar_type() == at::kInt && t->dim() == 1 && t->size(0) == s.batch + 1 && t->is_contiguous();
}
bool slopes_ok(const at::Tensor* t, const Shape& s) {
  return !t || (t->device() == s.device && t->scalar_type() == at::kFloat && t->dim() == 1 && t->size(0) == s.heads && t->is_contiguous());
}
bool words_ok(const at::Tensor* t, const Shape& s) {
  return !t || (t->device() == s.device && t->scalar_type() == at::kByte && t->is_contiguous());
}
bool bias_ok(const at::Tensor* t, const Shape& s, int64_t mq, int64_t mk) {  // what prepare_attn_bias() hands through
  if (!t) return true;
  return t->dim() == 4 && (t->size(0) == 1 || t->size(0) == s.batch) && (t->size(1) == 1 || t->size(1) == s.heads) && t->size(2) >= mq &&
         t->size(3) >= mk && t->device() == s.device && t->scalar_type() == s.dtype && t->stride(3) == 1 && t->stride(2) % 8 == 0 &&
         t->stride(2) >= mk && t->stride(0) % 8 == 0 && t->stride(1) % 8 == 0 && reinterpret_cast<uintptr_t>(ptr(*t)) % 16 == 0;
}
bool tables_ok(const at::Tensor* c, const at::Tensor* n, const Shape& s, int64_t rows) {
  if (!c && !n) return true;
  auto one = [&](const at::Tensor* t) {
    return t && t->dim() == 2 && t->size(1) == s.dim / 2 && t->scalar_type() == s.dtype && t->is_contiguous() && t->device() == s.device && t->size(0) >= rows;
  };
  return one(c) && one(n) && c->size(0) == n->size(0);
}
bool blocks_ok(const at::Tensor* m, const at::Tensor* order, const Shape& s, int32_t sq_r, int32_t sk_r) {
  if (!m) return true;
  if (!(m->is_cuda() && m->device() == s.device && m->scalar_type() == at::kInt && m->is_contiguous() && m->dim() == 2 && m->size(0) == sk_r / 256 && m->size(1) == sq_r / 16))
    return false;
  return !order || (order->device() == s.device && order->scalar_type() == at::kInt && order->is_contiguous() && order->numel() == sq_r / 16);
}

bool common(const at::Tensor* q, const at::Tensor* k, const at::Tensor* cu_q, Shape* s) {
  if (!g_bound || !q || !k || !cu_q || !q->is_cuda() || q->dim() != 3 || k->dim() != 3 || cu_q->dim() != 1) return false;
  s->dtype = q->scalar_type();
  if (s->dtype != at::kHalf && s->dtype != at::kBFloat16) return false;
  s->device = q->device();
  if (s->device.index() != c10::hip::current_device()) return false;
  s->total_q = q->size(0);
  s->total_k = k->size(0);
  s->heads = q->size(1);
  s->dim = q->size(2);
  s->batch = cu_q->size(0) - 1;
  return s->batch > 0 && (s->dim == 16 || s->dim == 32 || s->dim == 64 || s->dim == 128);
}
// (seed, offset) from a callable that draws them, called once nothing can be handed back to the binding any more; 0, 0 for None
bool draw(PyObject* f, uint64_t* seed, uint64_t* offset) {
  *seed = *offset = 0;
  if (f == Py_None) return true;
  PyObject* r = PyObject_CallNoArgs(f);
  if (!r) return false;
  if (PyTuple_Check(r) && PyTuple_GET_SIZE(r) == 2) {
    *seed = PyLong_AsUnsignedLongLong(PyTuple_GET_ITEM(r, 0));
    *offset = PyLong_AsUnsignedLongLong(PyTuple_GET_ITEM(r, 1));
  } else {
    PyErr_SetString(PyExc_TypeError, "(seed, offset) expected");
  }
  Py_DECREF(r);
  return !PyErr_Occurred();
}
PyObject* refused(int rc) { return PyErr_Format(PyExc_RuntimeError, "flash_attn_gfx950 error %d: %s", rc, g_lib.last_error()); }

// fwd(q, k, v, cu_q, cu_k, max_q, max_k, p, scale, zero, causal, draw, alibi, keep_words, bias, cos, sin, q_rot, blockmask, row_order)
// -> (out, softmax_lse) or None
PyObject* fwd(PyObject* const* a, Py_ssize_t n) {
  if (n != 20) return PyErr_Format(PyExc_TypeError, "fwd takes 20 arguments");
  bool ok = true;
  const at::Tensor *q = tensor(a[0], ok), *k = tensor(a[1], ok), *v = tensor(a[2], ok), *cu_q = tensor(a[3], ok), *cu_k = tensor(a[4], ok);
  const at::Tensor *alibi = tensor(a[12], ok), *words = tensor(a[13], ok), *bias = tensor(a[14], ok), *cos = tensor(a[15], ok), *sin = tensor(a[16], ok);
  const at::Tensor *q_rot = tensor(a[17], ok), *mask = tensor(a[18], ok), *order = tensor(a[19], ok);
  int64_t mq, mk;
  int32_t zero, causal;
  double p, scale;
  Shape s;
  if (!ok || !as_int(a[5], &mq) || !as_int(a[6], &mk) || !as_double(a[7], &p) || !as_double(a[8], &scale) || !as_flag(a[9], &zero) ||
      !as_flag(a[10], &causal) || mq <= 0 || mk <= 0 ||
      !common(q, k, cu_q, &s) || s.total_q > INT32_MAX || s.total_k > INT32_MAX || s.batch > INT32_MAX || !rows_ok(q, s, s.total_q) ||
      !rows_ok(k, s, s.total_k) || !rows_ok(v, s, s.total_k) || !cu_ok(cu_q, s) || !cu_ok(cu_k, s) || !slopes_ok(alibi, s) ||
      !words_ok(words, s) || !bias_ok(bias, s, mq, mk) || !tables_ok(cos, sin, s, mq) || (q_rot && (!cos || !rows_ok(q_rot, s, s.total_q))))
    Py_RETURN_NONE;
  int32_t sq_r, sk_r;
  g_lib.round_seqlens((int32_t)s.dim, (int32_t)mq, (int32_t)mk, mask != nullptr, &sq_r, &sk_r);
  if (!blocks_ok(mask, order, s, sq_r, sk_r)) Py_RETURN_NONE;

  at::Tensor o = at::empty({s.total_q, s.heads, s.dim}, q->options().memory_format(at::MemoryFormat::Contiguous).requires_grad(false));
  at::Tensor lse = at::empty({s.batch, s.heads, (int64_t)sq_r}, o.options().dtype(at::kFloat));
  fa_fwd_args f;
  memset(&f, 0, sizeof(f));
  f.struct_bytes = sizeof(f);
  f.dtype = s.dtype == at::kHalf ? FA_FP16 : FA_BF16;
  f.q = ptr(*q); f.k = ptr(*k); f.v = ptr(*v); f.o = ptr(o); f.softmax_lse = (float*)ptr(lse);
  f.cu_seqlens_q = (const int32_t*)ptr(*cu_q); f.cu_seqlens_k = (const int32_t*)ptr(*cu_k);
  f.q_row_stride = q->stride(0); f.q_head_stride = q->stride(1);
  f.k_row_stride = k->stride(0); f.k_head_stride = k->stride(1);
  f.v_row_stride = v->stride(0); f.v_head_stride = v->stride(1);
  f.o_row_stride = s.heads * s.dim; f.o_head_stride = s.dim;
  f.batch = (int32_t)s.batch; f.nheads = (int32_t)s.heads; f.head_dim = (int32_t)s.dim;
  f.total_q = (int32_t)s.total_q; f.total_k = (int32_t)s.total_k;
  f.max_seqlen_q = (int32_t)mq; f.max_seqlen_k = (int32_t)mk;
  f.p_dropout = (float)p; f.softmax_scale = (float)scale;
  f.zero_tensors = zero; f.is_causal = causal;
  if (alibi) f.alibi_slopes = (const float*)ptr(*alibi);
  if (words && !mask) { f.keep_words = ptr(*words); f.keep_words_bytes = (size_t)words->numel(); }
  if (bias) {
    f.attn_bias = ptr(*bias);
    f.bias_batch_stride = bias->size(0) == 1 ? 0 : bias->stride(0);
    f.bias_head_stride = bias->size(1) == 1 ? 0 : bias->stride(1);
    f.bias_row_stride = bias->stride(2);
  }
  if (cos) { f.rotary_cos = ptr(*cos); f.rotary_sin = ptr(*sin); f.rotary_table_rows = (int32_t)cos->size(0); }
  if (q_rot) { f.q_rot = ptr(*q_rot); f.q_rot_row_stride = q_rot->stride(0); f.q_rot_head_stride = q_rot->stride(1); }
  if (mask) { f.blockmask = (const int32_t*)ptr(*mask); if (order) f.row_order = (const int32_t*)ptr(*order); }
  at::Tensor ws;
  f.workspace_bytes = g_lib.fwd_workspace_bytes(&f);
  if (f.workspace_bytes) {
    ws = at::empty({(int64_t)f.workspace_bytes}, o.options().dtype(at::kByte));
    f.workspace = ptr(ws);
  }
  f.stream = c10::hip::getCurrentHIPStream(s.device.index()).stream();
  if (!draw(a[11], &f.philox_seed, &f.philox_offset)) return nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = (mask ? g_lib.fwd_block : g_lib.fwd)(&f);
  Py_END_ALLOW_THREADS
  if (rc != 0) return refused(rc);
  PyObject *po = THPVariable_Wrap(std::move(o)), *pl = THPVariable_Wrap(std::move(lse));
  PyObject* r = po && pl ? PyTuple_Pack(2, po, pl) : nullptr;
  Py_XDECREF(po);
  Py_XDECREF(pl);
  return r;
}

// bwd(dout, q, k, v, out, lse, dq, dk, dv, cu_q, cu_k, max_q, max_k, p, scale, zero, causal, draw, alibi, keep_words, bias, dbias, cos, sin,
// blockmask, row_order) -> softmax_d or None
PyObject* bwd(PyObject* const* a, Py_ssize_t n) {
  if (n != 26) return PyErr_Format(PyExc_TypeError, "bwd takes 26 arguments");
  bool ok = true;
  const at::Tensor* t[11];
  for (int i = 0; i < 11; i++) t[i] = tensor(a[i], ok);
  const at::Tensor *dout = t[0], *q = t[1], *k = t[2], *v = t[3], *out = t[4], *lse = t[5], *dq = t[6], *dk = t[7], *dv = t[8], *cu_q = t[9], *cu_k = t[10];
  const at::Tensor *alibi = tensor(a[18], ok), *words = tensor(a[19], ok), *bias = tensor(a[20], ok), *dbias = tensor(a[21], ok);
  const at::Tensor *cos = tensor(a[22], ok), *sin = tensor(a[23], ok), *mask = tensor(a[24], ok), *order = tensor(a[25], ok);
  int64_t mq, mk;
  int32_t zero, causal;
  double p, scale;
  Shape s;
  if (!ok || !as_int(a[11], &mq) || !as_int(a[12], &mk) || !as_double(a[13], &p) || !as_double(a[14], &scale) || !as_flag(a[15], &zero) ||
      !as_flag(a[16], &causal) || mq <= 0 || mk <= 0 ||
      !common(q, k, cu_q, &s) || s.total_q > INT32_MAX || s.total_k > INT32_MAX || s.batch > INT32_MAX || !rows_ok(q, s, s.total_q) ||
      !rows_ok(k, s, s.total_k) || !rows_ok(v, s, s.total_k) || !rows_ok(out, s, s.total_q) || !rows_ok(dout, s, s.total_q) ||
      !rows_ok(dq, s, s.total_q) || !rows_ok(dk, s, s.total_k) || !rows_ok(dv, s, s.total_k) || !out->is_contiguous() || !dout->is_contiguous() ||
      !cu_ok(cu_q, s) || !cu_ok(cu_k, s) || !lse || lse->device() != s.device || lse->scalar_type() != at::kFloat || lse->dim() != 3 ||
      lse->size(0) != s.batch || lse->size(1) != s.heads || lse->size(2) > INT32_MAX || !lse->is_contiguous() || !slopes_ok(alibi, s) ||
      !words_ok(words, s) || !bias_ok(bias, s, mq, mk) || !tables_ok(cos, sin, s, mq > mk ? mq : mk))
    Py_RETURN_NONE;
  if (dbias && !(bias && dbias->dim() == 4 && dbias->size(0) == s.batch && dbias->size(1) == s.heads && dbias->size(2) >= mq && dbias->size(3) >= mk &&
                 dbias->stride(3) == 1 && dbias->scalar_type() == s.dtype && dbias->device() == s.device))
    Py_RETURN_NONE;
  int32_t sq_r, sk_r;
  g_lib.round_seqlens((int32_t)s.dim, (int32_t)mq, (int32_t)mk, mask != nullptr, &sq_r, &sk_r);
  if (!blocks_ok(mask, order, s, sq_r, sk_r)) Py_RETURN_NONE;

  at::Tensor d = at::empty({s.batch, s.heads, (int64_t)sq_r}, lse->options().requires_grad(false));
  fa_bwd_args f;
  memset(&f, 0, sizeof(f));
  f.struct_bytes = sizeof(f);
  f.dtype = s.dtype == at::kHalf ? FA_FP16 : FA_BF16;
  f.dout = ptr(*dout); f.q = ptr(*q); f.k = ptr(*k); f.v = ptr(*v); f.out = ptr(*out); f.softmax_lse = (const float*)ptr(*lse);
  f.dq = ptr(*dq); f.dk = ptr(*dk); f.dv = ptr(*dv); f.softmax_d = (float*)ptr(d);
  f.cu_seqlens_q = (const int32_t*)ptr(*cu_q); f.cu_seqlens_k = (const int32_t*)ptr(*cu_k);
  f.do_row_stride = dout->stride(0); f.do_head_stride = dout->stride(1);
  f.q_row_stride = q->stride(0); f.q_head_stride = q->stride(1);
  f.k_row_stride = k->stride(0); f.k_head_stride = k->stride(1);
  f.v_row_stride = v->stride(0); f.v_head_stride = v->stride(1);
  f.o_row_stride = out->stride(0); f.o_head_stride = out->stride(1);
  f.dq_row_stride = dq->stride(0); f.dq_head_stride = dq->stride(1);
  f.dk_row_stride = dk->stride(0); f.dk_head_stride = dk->stride(1);
  f.dv_row_stride = dv->stride(0); f.dv_head_stride = dv->stride(1);
  f.lse_seq_stride = (int32_t)lse->size(2);
  f.batch = (int32_t)s.batch; f.nheads = (int32_t)s.heads; f.head_dim = (int32_t)s.dim;
  f.total_q = (int32_t)s.total_q; f.total_k = (int32_t)s.total_k;
  f.max_seqlen_q = (int32_t)mq; f.max_seqlen_k = (int32_t)mk;
  f.p_dropout = (float)p; f.softmax_scale = (float)scale;
  f.zero_tensors = zero; f.is_causal = causal;
  if (alibi) f.alibi_slopes = (const float*)ptr(*alibi);
  if (words && !mask) { f.keep_words = ptr(*words); f.keep_words_bytes = (size_t)words->numel(); }
  if (bias) {
    f.attn_bias = ptr(*bias);
    f.bias_batch_stride = bias->size(0) == 1 ? 0 : bias->stride(0);
    f.bias_head_stride = bias->size(1) == 1 ? 0 : bias->stride(1);
    f.bias_row_stride = bias->stride(2);
  }
  if (dbias) { f.dbias = ptr(*dbias); f.dbias_batch_stride = dbias->stride(0); f.dbias_head_stride = dbias->stride(1); f.dbias_row_stride = dbias->stride(2); }
  if (cos) { f.rotary_cos = ptr(*cos); f.rotary_sin = ptr(*sin); f.rotary_table_rows = (int32_t)cos->size(0); }
  if (mask) { f.blockmask = (const int32_t*)ptr(*mask); if (order) f.row_order = (const int32_t*)ptr(*order); }
  at::Tensor ws;
  f.workspace_bytes = g_lib.bwd_workspace_bytes(&f);
  if (f.workspace_bytes) {
    ws = at::empty({(int64_t)f.workspace_bytes}, q->options().memory_format(at::MemoryFormat::Contiguous).dtype(at::kByte).requires_grad(false));
    f.workspace = ptr(ws);
  }
  f.stream = c10::hip::getCurrentHIPStream(s.device.index()).stream();
  if (!draw(a[17], &f.philox_seed, &f.philox_offset)) return nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = (mask ? g_lib.bwd_block : g_lib.bwd)(&f);
  Py_END_ALLOW_THREADS
  if (rc != 0) return refused(rc);
  return THPVariable_Wrap(std::move(d));
}

// The calls around the attention itself: the keys' rotation, the copy of a bias with padded rows, the sum of its gradient.  us with the binding's
// own calls / with these: 14.3 / 4.1, 9.9 / 6.2 and 11.8 / 7.4 of the host's time for one; a step of 8 x 12 heads x 1024 with rotary 122.8 / 107.6 (kernels 107),
// of 8 x 8 x 421 .. 701 with a bias 151.6 / 124.6 (102).
hipStream_t stream_of(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
bool on_current_device(const at::Tensor* t) { return g_bound && t && t->is_cuda() && t->device().index() == c10::hip::current_device(); }
bool is_cu(const at::Tensor* t, const at::Tensor& like) {
  return t && t->is_cuda() && t->device() == like.device() && t->scalar_type() == at::kInt && t->dim() == 1 && t->size(0) > 1 && t->size(0) <= INT32_MAX &&
         t->is_contiguous();
}

// rotated_keys(qkv, cu, max_seqlen, cos, sin) -> (total, 2, nheads, headdim) with the rotated keys as part 1, or None
PyObject* rotated_keys(PyObject* const* a, Py_ssize_t n) {
  if (n != 5) return PyErr_Format(PyExc_TypeError, "rotated_keys takes 5 arguments");
  bool ok = true;
  const at::Tensor *qkv = tensor(a[0], ok), *cu = tensor(a[1], ok), *cos = tensor(a[3], ok), *sin = tensor(a[4], ok);
  int64_t ms;
  if (!ok || !as_int(a[2], &ms) || ms <= 0 || !on_current_device(qkv) || !is_cu(cu, *qkv) || !cos || !sin) Py_RETURN_NONE;
  const at::ScalarType type = qkv->scalar_type();
  if ((type != at::kHalf && type != at::kBFloat16) || qkv->dim() != 4 || qkv->size(0) <= 0 || qkv->size(0) > INT32_MAX || qkv->size(1) != 3 ||
      qkv->stride(3) != 1 || qkv->size(2) <= 0 || qkv->size(2) > INT32_MAX || qkv->size(3) <= 0 || qkv->size(3) % 8 != 0 || qkv->size(3) > INT32_MAX)
    Py_RETURN_NONE;
  const int64_t total = qkv->size(0), heads = qkv->size(2), dim = qkv->size(3), batch = cu->size(0) - 1;
  auto table = [&](const at::Tensor* t) {
    return t->dim() == 2 && t->size(1) == dim / 2 && t->scalar_type() == type && t->is_contiguous() && t->device() == qkv->device() && t->size(0) > 0 &&
           t->size(0) <= INT32_MAX && reinterpret_cast<uintptr_t>(ptr(*t)) % 8 == 0;
  };
  const bool ragged = total != batch * ms;
  if (!table(cos) || !table(sin) || cos->size(0) != sin->size(0) || (!ragged && cos->size(0) < ms)) Py_RETURN_NONE;
  const char* const k = static_cast<const char*>(ptr(*qkv)) + 2 * qkv->stride(1);
  if (reinterpret_cast<uintptr_t>(k) % 16 != 0 || qkv->stride(0) < 0 || qkv->stride(0) % 8 != 0 || qkv->stride(2) < 0 || qkv->stride(2) % 8 != 0 ||
      qkv->stride(1) < 0 || qkv->stride(1) % 8 != 0)
    Py_RETURN_NONE;
  at::Tensor rot = at::empty({total, 2, heads, dim}, qkv->options().memory_format(at::MemoryFormat::Contiguous).requires_grad(false)), pos;
  fa_rotary_args f;
  memset(&f, 0, sizeof(f));
  f.struct_bytes = sizeof(f);
  f.dtype = type == at::kHalf ? FA_FP16 : FA_BF16;
  f.src = k;
  f.dst = static_cast<char*>(ptr(rot)) + 2 * heads * dim;
  f.cos_table = ptr(*cos); f.sin_table = ptr(*sin);
  f.n_rows = total;
  f.src_row_stride = qkv->stride(0); f.src_part_stride = qkv->stride(1); f.src_head_stride = qkv->stride(2);
  f.dst_row_stride = 2 * heads * dim; f.dst_part_stride = heads * dim; f.dst_head_stride = dim;
  f.n_parts = f.n_rotated = 1;
  f.n_heads = (int32_t)heads; f.head_dim = (int32_t)dim;
  f.seqlen = (int32_t)ms; f.table_rows = (int32_t)cos->size(0);
  f.stream = stream_of(*qkv);
  if (ragged) {
    pos = at::empty({total}, cu->options().requires_grad(false));
    f.positions = (const int32_t*)ptr(pos);
  }
  int rc = 0;
  Py_BEGIN_ALLOW_THREADS
  if (ragged) rc = g_lib.token_positions((const int32_t*)ptr(*cu), (int32_t)batch, (int32_t)total, (int32_t*)ptr(pos), f.stream);
  if (rc == 0) rc = g_lib.rotary(&f);
  Py_END_ALLOW_THREADS
  return rc != 0 ? refused(rc) : THPVariable_Wrap(std::move(rot));
}

// pad_bias(bias): the copy with rows of a multiple of 8 keys that fa_fwd can read, or None
PyObject* pad_bias(PyObject* const* a, Py_ssize_t n) {
  if (n != 1) return PyErr_Format(PyExc_TypeError, "pad_bias takes 1 argument");
  bool ok = true;
  const at::Tensor* t = tensor(a[0], ok);
  if (!ok || !on_current_device(t) || (t->scalar_type() != at::kHalf && t->scalar_type() != at::kBFloat16) || t->dim() != 4 || t->size(0) > INT32_MAX ||
      t->size(1) > INT32_MAX)
    Py_RETURN_NONE;
  at::Tensor out = at::empty({t->size(0), t->size(1), t->size(2), (t->size(3) + 7) / 8 * 8},
                             t->options().memory_format(at::MemoryFormat::Contiguous).requires_grad(false));
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_lib.pad_bias_rows(ptr(*t), ptr(out), (int32_t)t->size(0), (int32_t)t->size(1), t->size(2), t->size(3), t->stride(0), t->stride(1), t->stride(2),
                           t->stride(3), stream_of(*t));
  Py_END_ALLOW_THREADS
  return rc != 0 ? refused(rc) : THPVariable_Wrap(std::move(out));
}

// reduce_bias_grad(dbias, out, sum_batch, sum_heads, cu_q, cu_k, total_q, total_k, causal) -> True or None
PyObject* reduce_bias_grad(PyObject* const* a, Py_ssize_t n) {
  if (n != 9) return PyErr_Format(PyExc_TypeError, "reduce_bias_grad takes 9 arguments");
  bool ok = true;
  const at::Tensor *d = tensor(a[0], ok), *o = tensor(a[1], ok), *cu_q = tensor(a[4], ok), *cu_k = tensor(a[5], ok);
  int32_t sum_b, sum_h, causal;
  int64_t tq, tk;
  if (!ok || !on_current_device(d) || !o || !as_flag(a[2], &sum_b) || !as_flag(a[3], &sum_h) || !as_int(a[6], &tq) || !as_int(a[7], &tk) ||
      !as_flag(a[8], &causal) || (d->scalar_type() != at::kHalf && d->scalar_type() != at::kBFloat16) || d->dim() != 4 || o->dim() != 4 ||
      o->device() != d->device() || o->scalar_type() != d->scalar_type() || !is_cu(cu_q, *d) || !is_cu(cu_k, *d))
    Py_RETURN_NONE;
  const int64_t batch = d->size(0), heads = d->size(1), rows = d->size(2), cols = o->size(3);
  if (o->size(0) != (sum_b ? 1 : batch) || o->size(1) != (sum_h ? 1 : heads) || o->size(2) != rows || cols > d->size(3) || d->stride(3) != 1 ||
      (o->stride(3) != 1 && cols > 1) || cu_q->size(0) != batch + 1 || cu_k->size(0) != batch + 1 || heads > INT32_MAX || rows > INT32_MAX ||
      cols > INT32_MAX)
    Py_RETURN_NONE;
  fa_bwd_args f;
  memset(&f, 0, sizeof(f));
  f.struct_bytes = sizeof(f);
  f.dtype = d->scalar_type() == at::kHalf ? FA_FP16 : FA_BF16;
  f.batch = (int32_t)batch; f.nheads = (int32_t)heads;
  f.total_q = (int32_t)tq; f.total_k = (int32_t)tk;
  f.max_seqlen_q = (int32_t)rows; f.max_seqlen_k = (int32_t)cols;
  f.cu_seqlens_q = (const int32_t*)ptr(*cu_q); f.cu_seqlens_k = (const int32_t*)ptr(*cu_k);
  f.is_causal = causal;
  f.dbias_batch_stride = d->stride(0); f.dbias_head_stride = d->stride(1); f.dbias_row_stride = d->stride(2);
  f.stream = stream_of(*d);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_lib.bias_grad_reduce_ragged(ptr(*d), ptr(*o), &f, sum_b, sum_h, o->stride(0), o->stride(1), o->stride(2));
  Py_END_ALLOW_THREADS
  if (rc != 0) return refused(rc);
  Py_RETURN_TRUE;
}

// C++ exceptions (an allocation that fails, memory that may not be touched under tracing) do not leave the module: the call is handed back and
// the binding meets the same condition
template <PyObject* (*F)(PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject*, PyObject* const* a, Py_ssize_t n) {
  try {
    return F(a, n);
  } catch (const std::exception&) {
    if (PyErr_Occurred()) return nullptr;
    Py_RETURN_NONE;
  }
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void (*)(void))py_bind, METH_FASTCALL, nullptr},
    {"fwd", (PyCFunction)(void (*)(void))guarded<fwd>, METH_FASTCALL, nullptr},
    {"bwd", (PyCFunction)(void (*)(void))guarded<bwd>, METH_FASTCALL, nullptr},
    {"rotated_keys", (PyCFunction)(void (*)(void))guarded<rotated_keys>, METH_FASTCALL, nullptr},
    {"pad_bias", (PyCFunction)(void (*)(void))guarded<pad_bias>, METH_FASTCALL, nullptr},
    {"reduce_bias_grad", (PyCFunction)(void (*)(void))guarded<reduce_bias_grad>, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "fa_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_fa_host() { return PyModule_Create(&module); }
