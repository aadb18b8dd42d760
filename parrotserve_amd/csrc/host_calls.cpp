// The wrappers of kernels.py for the calls a decoder layer makes, in C++: the argument checks, the result's allocation
// and the call into the C ABI, without the interpreter between them.  Each function takes the plain form of its call --
// exact torch tensors on one GPU, dense in their last dimension, 16- or 32-bit floating point -- and returns None for
// everything else: the Python body then decides, and raises what it always raised.  Nothing is kept between calls.
//
// Bound by the launches: a kernel launch takes 3.4 us of host time on an MI355X host, and a decode batch of a few
// requests needs less than that of the device per kernel.  In Python what stood around the launches took another 3.9 us
// for a norm, 5.3 for rotary + append, 8.0 for decode attention, 4.5 for add + norm and 4.0 for the activation (reading
// a tensor's attributes costs 0.1 us each, and there are ten to forty of them).  A layer's own kernels for 8 requests
// over 512 tokens, issued one after the other: 49.1 us in Python, 31 to 32 here, 28 of them on the device.
#include <Python.h>

#include <ATen/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cmath>
#include <cstring>

#include "../../include/parrot_hip.h"

namespace {

#define PH_ENTRIES(X)                                                                                        \
  X(ph_rms_norm) X(ph_add_rms_norm) X(ph_silu_mul) X(ph_rope_append) X(ph_sample_top_p) X(ph_decode_attention) \
  X(ph_decode_attention_gqa) X(ph_prefill_attention) X(ph_prefill_workspace_bytes) X(ph_prefill_workspace_min_bytes)

// addresses of the library's entry points, given by bind() (the profiling variant of the library has other ones)
struct Entries {
#define X(fn) decltype(&::fn) fn = nullptr;
  PH_ENTRIES(X)
#undef X
} lib;

// what the Python module keeps its state in, given by bind()
struct Module {
  PyObject *check, *raw_stream, *raw_device, *capturing, *workspaces, *workspace, *decode_workspace_bytes,
      *decode_tables, *prefill_tables;
} py;

// attribute names of the table classes
struct Names {
  PyObject *num_reqs, *num_groups, *prefix_slots, *prefix_cu, *group_req_cu, *group_req_cu_host, *max_prefix_len,
      *suffix_slots, *suffix_offsets, *suffix_table_stride, *suffix_lens, *max_suffix_len, *chunk_tokens, *plan,
      *suffix_slots_count, *num_tokens, *num_chunks, *q_cu, *kv_cu, *ctx_slots, *max_kv_len;
} name;

struct Ref {  // an owned reference
  PyObject* p;
  explicit Ref(PyObject* q = nullptr) : p(q) {}
  Ref(const Ref&) = delete;
  ~Ref() { Py_XDECREF(p); }
  operator PyObject*() const { return p; }
};

// A tensor of exactly torch's own class that owns memory on a GPU (no subclass, no wrapper of a transform); null: not plain.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage() || t.is_conj() || t.is_neg() ||
      t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                               c10::DispatchKey::Functionalize, c10::DispatchKey::Python})))
    return nullptr;
  return &t;
}

int dtype_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kHalf: return PH_F16;
    case at::kBFloat16: return PH_BF16;
    case at::kFloat: return PH_F32;
    default: return -1;
  }
}

bool same_kind(const at::Tensor& a, const at::Tensor& b) {
  return a.device() == b.device() && a.scalar_type() == b.scalar_type();
}

// [rows, n] whose rows are dense
bool is_rows(const at::Tensor& t) { return t.dim() == 2 && t.numel() > 0 && t.stride(1) == 1; }
// [n, heads, dim] whose tokens' heads are dense rows
bool is_heads(const at::Tensor& t) {
  return t.dim() == 3 && t.numel() > 0 && t.stride(2) == 1 && t.stride(1) == t.size(2);
}

bool number(PyObject* o, double& v) {
  if (PyFloat_CheckExact(o)) v = PyFloat_AS_DOUBLE(o);
  else if (PyLong_CheckExact(o)) v = PyLong_AsDouble(o);
  else return false;
  if (v == -1.0 && PyErr_Occurred()) {  // beyond a double: the Python body's to refuse
    PyErr_Clear();
    return false;
  }
  return true;
}

bool whole(PyObject* o, int64_t& v) {
  if (!o || !(PyLong_CheckExact(o) || PyBool_Check(o))) return false;
  v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

bool int_of(PyObject* obj, PyObject* attr, int64_t& v) {
  Ref r(PyObject_GetAttr(obj, attr));
  if (!r.p) PyErr_Clear();
  return whole(r.p, v);
}

// address of a table's tensor, null for None; false: neither a plain tensor nor None
template <typename T>
bool addr_of(PyObject* obj, PyObject* attr, T*& v, const at::Tensor** tensor = nullptr, bool on_host = false) {
  Ref r(PyObject_GetAttr(obj, attr));
  if (!r.p) {
    PyErr_Clear();
    return false;
  }
  v = nullptr;
  if (r.p == Py_None) return true;
  if (on_host ? !THPVariable_CheckExact(r) : !plain(r)) return false;
  const at::Tensor& t = THPVariable_Unpack(r.p);  // (the table holds the tensor for the length of the call)
  if (on_host && (!t.has_storage() || !t.is_cpu())) return false;
  v = static_cast<T*>(t.data_ptr());
  if (tensor) *tensor = &t;
  return true;
}

// torch's current stream of the current device, as kernels._stream gives it; false with an error set
bool current_stream(int64_t& device, void*& stream, PyObject** stream_obj = nullptr) {
  Ref dev(PyObject_CallNoArgs(py.raw_device));
  if (!dev.p) return false;
  device = PyLong_AsLongLong(dev);
  PyObject* st = PyObject_CallOneArg(py.raw_stream, dev);
  if (!st) return false;
  stream = PyLong_AsVoidPtr(st);
  if (stream_obj) *stream_obj = st;
  else Py_DECREF(st);
  return !PyErr_Occurred();
}

// kernels._workspace: the stream's buffer where it is large enough and nothing is being captured, else that function's
// own doing.  `keep` holds the buffer for the length of the call.
bool workspace(int64_t nbytes, const at::Tensor& like, PyObject* stream_obj, PyObject* least, Ref& keep, void*& ptr,
               int64_t& size) {
  Ref capturing(PyObject_CallNoArgs(py.capturing));
  if (!capturing.p) return false;
  if (capturing.p == Py_False) {
    const int index = like.device().index();
    Ref key(Py_BuildValue("(iO)", index < 0 ? 0 : index, stream_obj));
    if (!key.p) return false;
    PyObject* buf = PyDict_GetItemWithError(py.workspaces, key);
    if (!buf && PyErr_Occurred()) return false;
    if (buf && THPVariable_Check(buf) && THPVariable_Unpack(buf).numel() >= nbytes) {
      Py_INCREF(buf);
      keep.p = buf;
    }
  }
  if (!keep.p) {
    Ref dev(THPVariable_Wrap(like));
    Ref device(dev.p ? PyObject_GetAttrString(dev, "device") : nullptr);
    if (!device.p) return false;
    keep.p = least ? PyObject_CallFunction(py.workspace, "LOO", (long long)nbytes, device.p, least)
                   : PyObject_CallFunction(py.workspace, "LO", (long long)nbytes, device.p);
    if (!keep.p) return false;
  }
  const at::Tensor& t = THPVariable_Unpack(keep.p);
  ptr = t.data_ptr();
  size = t.numel();
  return true;
}

// the launch itself runs without the interpreter's lock, as it does through ctypes
template <typename F>
int unlocked(F f) {
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = f();
  Py_END_ALLOW_THREADS
  return rc;
}

PyObject* result(int rc, const char* what, const at::Tensor& out) {
  if (rc != PH_OK) {
    Ref r(PyObject_CallFunction(py.check, "is", rc, what));
    return nullptr;
  }
  return THPVariable_Wrap(out);
}

at::Tensor dense_like(const at::Tensor& t) {
  return at::empty_like(t, t.options(), at::MemoryFormat::Contiguous);
}

// rms_norm(x, weight, eps, round_first, what)
PyObject* rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5) Py_RETURN_NONE;
  const at::Tensor *x = plain(a[0]), *w = plain(a[1]);
  double eps;
  int64_t first;
  if (!x || !w || !is_rows(*x) || w->dim() != 1 || w->size(0) != x->size(1) || !w->is_contiguous() ||
      !same_kind(*x, *w) || dtype_code(*x) < 0 || !number(a[2], eps) || !whole(a[3], first))
    Py_RETURN_NONE;
  const char* what = PyUnicode_AsUTF8(a[4]);
  int64_t dev;
  void* st;
  if (!what || !current_stream(dev, st)) return nullptr;
  const at::Tensor out = dense_like(*x);
  void *o = out.data_ptr(), *xp = x->data_ptr(), *wp = w->data_ptr();
  const int rc = unlocked([&] {
    return lib.ph_rms_norm(o, xp, wp, (float)eps, x->size(0), x->size(1), x->stride(0), x->size(1), dtype_code(*x),
                           (int)first, st);
  });
  return result(rc, what, out);
  END_HANDLE_TH_ERRORS
}

// add_rms_norm(x, residual, weight, eps, round_first)
PyObject* add_rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5) Py_RETURN_NONE;
  const at::Tensor *x = plain(a[0]), *r = plain(a[1]), *w = plain(a[2]);
  double eps;
  int64_t first;
  if (!x || !r || !w || !is_rows(*x) || !is_rows(*r) || x->sizes() != r->sizes() || w->dim() != 1 ||
      w->size(0) != x->size(1) || !w->is_contiguous() || !same_kind(*x, *w) || !same_kind(*x, *r) ||
      dtype_code(*x) < 0 || !number(a[3], eps) || !whole(a[4], first))
    Py_RETURN_NONE;
  int64_t dev;
  void* st;
  if (!current_stream(dev, st)) return nullptr;
  const at::Tensor out = dense_like(*x);
  void *o = out.data_ptr(), *rp = r->data_ptr(), *xp = x->data_ptr(), *wp = w->data_ptr();
  const int rc = unlocked([&] {
    return lib.ph_add_rms_norm(o, rp, xp, wp, (float)eps, x->size(0), x->size(1), x->stride(0), r->stride(0),
                               x->size(1), dtype_code(*x), first ? 1 : 0, st);
  });
  return result(rc, "fused_add_rms_norm", out);
  END_HANDLE_TH_ERRORS
}

// silu_mul(gate, up)
PyObject* silu_mul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2) Py_RETURN_NONE;
  const at::Tensor *g = plain(a[0]), *u = plain(a[1]);
  if (!g || !u || !is_rows(*g) || !is_rows(*u) || g->sizes() != u->sizes() || !same_kind(*g, *u) || dtype_code(*g) < 0)
    Py_RETURN_NONE;
  int64_t dev;
  void* st;
  if (!current_stream(dev, st)) return nullptr;
  const at::Tensor out = dense_like(*g);
  void *o = out.data_ptr(), *gp = g->data_ptr(), *up = u->data_ptr();
  const int rc = unlocked([&] {
    return lib.ph_silu_mul(o, gp, up, g->size(0), g->size(1), g->stride(0), u->stride(0), g->size(1), dtype_code(*g),
                           st);
  });
  return result(rc, "silu_mul", out);
  END_HANDLE_TH_ERRORS
}

// rope_append(positions, query, key, value, cos_sin, head_size, key_cache, value_cache, slots, key_in_place) -> True
PyObject* rope_append(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 10) Py_RETURN_NONE;
  const at::Tensor *pos = plain(a[0]), *q = plain(a[1]), *k = plain(a[2]), *v = plain(a[3]), *cs = plain(a[4]),
                   *kc = plain(a[6]), *vc = plain(a[7]), *slots = plain(a[8]);
  int64_t D, in_place;
  if (!pos || !q || !k || !v || !cs || !kc || !vc || !slots || !whole(a[5], D) || D <= 0 || !whole(a[9], in_place))
    Py_RETURN_NONE;
  const int code = dtype_code(*q);
  if (code < 0 || pos->scalar_type() != at::kLong || pos->dim() != 1 || !pos->is_contiguous() || !is_rows(*q) ||
      !is_rows(*k) || !is_rows(*v) || !is_heads(*kc) || !is_heads(*vc) || cs->dim() < 1 || !cs->is_contiguous() ||
      !slots->is_contiguous() || pos->device() != q->device() || slots->device() != q->device() ||
      (slots->scalar_type() != at::kInt && slots->scalar_type() != at::kLong))
    Py_RETURN_NONE;
  const int64_t T = pos->size(0), hq = q->size(1) / D, hk = k->size(1) / D;
  if (!same_kind(*q, *k) || !same_kind(*q, *v) || !same_kind(*q, *kc) || !same_kind(*q, *vc) || !same_kind(*q, *cs) ||
      q->size(0) != T || k->size(0) != T || v->size(0) != T || v->size(1) != hk * D || kc->size(1) != hk ||
      kc->size(2) != D || vc->size(1) != hk || vc->size(2) != D || kc->stride(0) != vc->stride(0) ||
      slots->numel() != T)
    Py_RETURN_NONE;
  int64_t dev;
  void* st;
  if (!current_stream(dev, st)) return nullptr;
  const int64_t* pp = static_cast<const int64_t*>(pos->data_ptr());
  void *qp = q->data_ptr(), *kp = k->data_ptr(), *vp = v->data_ptr(), *cp = cs->data_ptr(), *kcp = kc->data_ptr(),
       *vcp = vc->data_ptr(), *sp = slots->data_ptr();
  const int idx = slots->scalar_type() == at::kInt ? PH_IDX_I32 : PH_IDX_I64;
  const int rc = unlocked([&] {
    return lib.ph_rope_append(pp, qp, kp, vp, cp, kcp, vcp, sp, idx, T, hq, hk, D, cs->size(-1), q->stride(0),
                              k->stride(0), v->stride(0), kc->stride(0), code, in_place ? 1 : 0, st);
  });
  if (rc != PH_OK) {
    Ref r(PyObject_CallFunction(py.check, "is", rc, "rope_and_cache"));
    return nullptr;
  }
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// sample_top_p(logits, temperature, top_p, uniform)
PyObject* sample_top_p(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4) Py_RETURN_NONE;
  const at::Tensor* x = plain(a[0]);
  if (!x || !is_rows(*x) || dtype_code(*x) < 0) Py_RETURN_NONE;
  const int64_t B = x->size(0), V = x->size(1);
  const float* row[3] = {nullptr, nullptr, nullptr};
  for (int i = 0; i < 3; ++i) {
    if (i < 2 && a[1 + i] == Py_None) continue;
    const at::Tensor* t = plain(a[1 + i]);
    if (!t || t->device() != x->device() || t->scalar_type() != at::kFloat || t->numel() != B || !t->is_contiguous())
      Py_RETURN_NONE;
    row[i] = static_cast<const float*>(t->data_ptr());
  }
  int64_t dev;
  void* st;
  if (!current_stream(dev, st)) return nullptr;
  const at::Tensor out = at::empty({B}, x->options().dtype(at::kLong));
  int64_t* o = static_cast<int64_t*>(out.data_ptr());
  void* xp = x->data_ptr();
  const int64_t stride = B > 1 ? x->stride(0) : std::max<int64_t>(x->stride(0), V);
  const int rc = unlocked(
      [&] { return lib.ph_sample_top_p(xp, stride, row[0], row[1], row[2], o, B, V, dtype_code(*x), st); });
  return result(rc, "sample_top_p", out);
  END_HANDLE_TH_ERRORS
}

// the caches of an attention call: [slots, kv heads, dim], alike, of the query's kind
bool are_caches(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v) {
  return is_heads(q) && is_heads(k) && k.sizes() == v.sizes() && k.strides() == v.strides() && same_kind(q, k) &&
         same_kind(q, v) && q.size(2) == k.size(2) && dtype_code(q) >= 0;
}

bool scale_of(PyObject* o, int64_t D, float& scale) {
  double s = std::pow((double)D, -0.5);
  if (o != Py_None && !number(o, s)) return false;
  scale = (float)s;
  return true;
}

// decode_attention(query, key_cache, value_cache, tables, scale, head_mapping, kv_group)
PyObject* decode_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 7) Py_RETURN_NONE;
  const at::Tensor *q = plain(a[0]), *k = plain(a[1]), *v = plain(a[2]);
  PyObject* t = a[3];
  float scale;
  int64_t kv_group;
  if (!q || !k || !v || (PyObject*)Py_TYPE(t) != py.decode_tables || !are_caches(*q, *k, *v) ||
      !scale_of(a[4], q->size(2), scale) || !whole(a[6], kv_group))
    Py_RETURN_NONE;
  const int64_t B = q->size(0), H = q->size(1), D = q->size(2);
  const int32_t* map = nullptr;
  if (a[5] != Py_None) {
    const at::Tensor* m = plain(a[5]);
    if (!m || m->scalar_type() != at::kInt || m->numel() != H || !m->is_contiguous() || m->device() != q->device())
      Py_RETURN_NONE;
    map = static_cast<const int32_t*>(m->data_ptr());
  } else if (k->size(1) != H) {
    Py_RETURN_NONE;
  }
  int64_t reqs, groups, max_prefix, max_suffix, chunk, table_stride;
  const int32_t *p_slots, *p_cu, *g_cu, *g_cu_host, *s_slots, *s_lens;
  const int64_t* s_off;
  const at::Tensor* table = nullptr;
  if (!int_of(t, name.num_reqs, reqs) || reqs != B || !int_of(t, name.num_groups, groups) ||
      !int_of(t, name.max_prefix_len, max_prefix) || !int_of(t, name.max_suffix_len, max_suffix) ||
      !int_of(t, name.chunk_tokens, chunk) || !int_of(t, name.suffix_table_stride, table_stride) ||
      !addr_of(t, name.prefix_slots, p_slots) || !addr_of(t, name.prefix_cu, p_cu) ||
      !addr_of(t, name.group_req_cu, g_cu) || !addr_of(t, name.group_req_cu_host, g_cu_host, nullptr, true) ||
      !addr_of(t, name.suffix_slots, s_slots, &table) || !addr_of(t, name.suffix_offsets, s_off) ||
      !addr_of(t, name.suffix_lens, s_lens))
    Py_RETURN_NONE;
  // DecodeTables.suffix_slots_count (an instance may carry its own)
  Ref own(PyObject_GenericGetDict(t, nullptr));
  if (!own.p || PyDict_Contains(own, name.suffix_slots_count) != 0) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  int64_t s_count = 0;
  if (table && s_off) s_count = table->numel();
  else if (table && table->dim() < 1) Py_RETURN_NONE;
  else if (table) s_count = (reqs - 1) * table_stride + table->size(-1);
  ph_suffix_plan plan_copy;
  const ph_suffix_plan* plan = nullptr;
  Ref plan_obj(PyObject_GetAttr(t, name.plan));
  if (!plan_obj.p) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  if (plan_obj.p != Py_None) {
    Py_buffer view;
    if (PyObject_GetBuffer(plan_obj, &view, PyBUF_SIMPLE) != 0) {
      PyErr_Clear();
      Py_RETURN_NONE;
    }
    const bool fits = view.len == (Py_ssize_t)sizeof(plan_copy);
    if (fits) std::memcpy(&plan_copy, view.buf, sizeof(plan_copy));
    PyBuffer_Release(&view);
    if (!fits) Py_RETURN_NONE;
    plan = &plan_copy;
  }
  int64_t dev, ws_bytes;
  void *st, *ws;
  PyObject* stream_obj = nullptr;
  if (!current_stream(dev, st, &stream_obj)) return nullptr;
  Ref stream_ref(stream_obj), keep;
  Ref need(PyObject_CallFunction(py.decode_workspace_bytes, "LLLLLLLLL", (long long)dev, (long long)B, (long long)H,
                                 (long long)D, (long long)groups, (long long)max_prefix, (long long)max_suffix,
                                 (long long)chunk, (long long)(plan ? plan->num_items : 0)));
  if (!need.p) return nullptr;
  const at::Tensor out = dense_like(*q);
  if (!workspace(PyLong_AsLongLong(need), *q, stream_obj, nullptr, keep, ws, ws_bytes)) return nullptr;
  void *o = out.data_ptr(), *qp = q->data_ptr(), *kp = k->data_ptr(), *vp = v->data_ptr();
  const int code = dtype_code(*q);
  const int rc = unlocked([&] {
    return map ? lib.ph_decode_attention_gqa(o, qp, kp, vp, B, H, k->size(1), map, kv_group, D, code, q->stride(0),
                                             H * D, k->stride(0), scale, groups, p_slots, p_cu, g_cu, g_cu_host,
                                             max_prefix, s_slots, s_off, table_stride, s_count, s_lens, max_suffix,
                                             chunk, plan, ws, (size_t)ws_bytes, st)
               : lib.ph_decode_attention(o, qp, kp, vp, B, H, D, code, q->stride(0), H * D, k->stride(0), scale, groups,
                                         p_slots, p_cu, g_cu, g_cu_host, max_prefix, s_slots, s_off, table_stride,
                                         s_count, s_lens, max_suffix, chunk, plan, ws, (size_t)ws_bytes, st);
  });
  return result(rc, "decode_attention", out);
  END_HANDLE_TH_ERRORS
}

// prefill_attention(query, key_cache, value_cache, tables, scale)
PyObject* prefill_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5) Py_RETURN_NONE;
  const at::Tensor *q = plain(a[0]), *k = plain(a[1]), *v = plain(a[2]);
  PyObject* t = a[3];
  float scale;
  if (!q || !k || !v || (PyObject*)Py_TYPE(t) != py.prefill_tables || !are_caches(*q, *k, *v) ||
      k->size(1) != q->size(1) || !scale_of(a[4], q->size(2), scale))
    Py_RETURN_NONE;
  const int64_t T = q->size(0), H = q->size(1), D = q->size(2);
  int64_t tokens, chunks, max_kv;
  const int32_t *q_cu, *kv_cu, *slots;
  const at::Tensor* slots_t = nullptr;
  if (!int_of(t, name.num_tokens, tokens) || tokens != T || !int_of(t, name.num_chunks, chunks) ||
      !int_of(t, name.max_kv_len, max_kv) || !addr_of(t, name.q_cu, q_cu) || !addr_of(t, name.kv_cu, kv_cu) ||
      !addr_of(t, name.ctx_slots, slots, &slots_t) || !slots_t)
    Py_RETURN_NONE;
  const int code = dtype_code(*q);
  int64_t dev, ws_bytes;
  void *st, *ws;
  PyObject* stream_obj = nullptr;
  if (!current_stream(dev, st, &stream_obj)) return nullptr;
  Ref stream_ref(stream_obj), keep;
  const at::Tensor out = at::empty({T, H, D}, q->options());
  Ref least(PyLong_FromSize_t(lib.ph_prefill_workspace_min_bytes(T, H, D, code, max_kv)));
  if (!least.p || !workspace((int64_t)lib.ph_prefill_workspace_bytes(T, H, D, code, max_kv), *q, stream_obj, least,
                             keep, ws, ws_bytes))
    return nullptr;
  void *o = out.data_ptr(), *qp = q->data_ptr(), *kp = k->data_ptr(), *vp = v->data_ptr();
  const int64_t n_slots = slots_t->numel();
  const int rc = unlocked([&] {
    return lib.ph_prefill_attention(o, qp, kp, vp, T, chunks, H, D, code, q->stride(0), H * D, k->stride(0), scale,
                                    q_cu, kv_cu, slots, n_slots, max_kv, ws, (size_t)ws_bytes, st);
  });
  return result(rc, "prefill_attention", out);
  END_HANDLE_TH_ERRORS
}

// bind({entry point: address}, {name: object of the Python module})
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 2 || !PyDict_Check(a[0]) || !PyDict_Check(a[1])) {
    PyErr_SetString(PyExc_TypeError, "bind(entries, module objects)");
    return nullptr;
  }
#define X(fn)                                                                      \
  {                                                                                \
    PyObject* v = PyDict_GetItemString(a[0], #fn);                                 \
    void* p = v ? PyLong_AsVoidPtr(v) : nullptr;                                   \
    if (!p) return PyErr_Format(PyExc_KeyError, "no address for %s", #fn);         \
    lib.fn = reinterpret_cast<decltype(lib.fn)>(p);                                \
  }
  PH_ENTRIES(X)
#undef X
#define X(field)                                                                   \
  {                                                                                \
    PyObject* v = PyDict_GetItemString(a[1], #field);                              \
    if (!v) return PyErr_Format(PyExc_KeyError, "no object for %s", #field);       \
    Py_INCREF(v);                                                                  \
    Py_XSETREF(py.field, v);                                                       \
  }
  X(check) X(raw_stream) X(raw_device) X(capturing) X(workspaces) X(workspace) X(decode_workspace_bytes)
  X(decode_tables) X(prefill_tables)
#undef X
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
#define X(fn, doc) {#fn, (PyCFunction)(void (*)(void))fn, METH_FASTCALL, doc},
    X(bind, "bind(entries, objects): addresses of the library and objects of the Python module")
    X(rms_norm, "rms_norm(x, weight, eps, round_first, what) -> tensor, or None: not the plain form")
    X(add_rms_norm, "add_rms_norm(x, residual, weight, eps, round_first) -> tensor or None")
    X(silu_mul, "silu_mul(gate, up) -> tensor or None")
    X(rope_append, "rope_append(positions, q, k, v, cos_sin, head_size, k_cache, v_cache, slots, in_place) -> True or None")
    X(sample_top_p, "sample_top_p(logits, temperature, top_p, uniform) -> tensor or None")
    X(decode_attention, "decode_attention(q, k, v, tables, scale, head_mapping, kv_group) -> tensor or None")
    X(prefill_attention, "prefill_attention(q, k, v, tables, scale) -> tensor or None")
#undef X
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "kernels.py's plain calls in C++", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
#define X(field) \
  if (!(name.field = PyUnicode_InternFromString(#field))) return nullptr;
  X(num_reqs) X(num_groups) X(prefix_slots) X(prefix_cu) X(group_req_cu) X(group_req_cu_host) X(max_prefix_len)
  X(suffix_slots) X(suffix_offsets) X(suffix_table_stride) X(suffix_lens) X(max_suffix_len) X(chunk_tokens) X(plan)
  X(suffix_slots_count) X(num_tokens) X(num_chunks) X(q_cu) X(kv_cu) X(ctx_slots) X(max_kv_len)
#undef X
  return PyModule_Create(&module);
}
