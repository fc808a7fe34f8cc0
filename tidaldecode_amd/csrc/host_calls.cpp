// The regular case of the Python entry points' host work, in one native call each: the checks of
// _kernels.py on the tensors, the argument structures, the plan, and the call into libtidal_hip.so.
//
// A decode step of a short context is bound by its host: a Python entry point spends 8 to 14 us in
// tensor attribute reads, ctypes structures and argument conversion for a kernel of 5 us.  Every
// function here returns True, or the output it made, after it has launched, and False, having launched nothing, for
// whatever it does not recognise as regular (an argument of another kind, a check that fails, a handle's workspace
// that has to grow): the caller then goes on in Python, which raises the errors and handles the
// rest.  Nothing is kept between calls; the only state is the table of function addresses.
#include <Python.h>
#include <ATen/ATen.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>

#include "../../include/tidal_hip.h"

namespace {

struct Lib {
  decltype(&td_last_error) last_error;
  decltype(&td_decode_make_plan) make_plan;
  decltype(&td_short_list_pays) short_list_pays;
  decltype(&td_decode_attn) decode_attn;
  decltype(&td_decode_attn_noalloc) decode_attn_noalloc;
  decltype(&td_topk_segments) topk_segments;
  decltype(&td_topk_workspace_bytes) topk_workspace_bytes;
  decltype(&td_rope_table) rope_table;
  decltype(&td_rope_in_place) rope_in_place;
  decltype(&td_append_kv) append_kv;
  decltype(&td_prefill_workspace_bytes) prefill_workspace_bytes;
  decltype(&td_prefill_attn_split) prefill_attn_split;
  decltype(&td_gemv) gemv;
  decltype(&td_score_reduce) score_reduce;
  decltype(&td_estimate_score) estimate_score;
} lib;

template <typename F>
bool take(PyObject* table, const char* name, F& fn) {
  PyObject* v = PyDict_GetItemString(table, name);
  if (!v) {
    PyErr_Format(PyExc_KeyError, "%s", name);
    return false;
  }
  fn = reinterpret_cast<F>(PyLong_AsVoidPtr(v));
  return fn != nullptr;
}

PyObject* bind(PyObject*, PyObject* table) {
  if (!PyDict_Check(table)) Py_RETURN_FALSE;
#define TD_TAKE(f) \
  if (!take(table, "td_" #f, lib.f)) return nullptr;
  TD_TAKE(last_error)
  TD_TAKE(short_list_pays)
  TD_TAKE(decode_attn)
  TD_TAKE(decode_attn_noalloc)
  TD_TAKE(topk_segments)
  TD_TAKE(topk_workspace_bytes)
  TD_TAKE(rope_table)
  TD_TAKE(rope_in_place)
  TD_TAKE(append_kv)
  TD_TAKE(prefill_workspace_bytes)
  TD_TAKE(prefill_attn_split)
  TD_TAKE(gemv)
  TD_TAKE(score_reduce)
  TD_TAKE(estimate_score)
#undef TD_TAKE
  if (!take(table, "td_decode_make_plan", lib.make_plan)) return nullptr;
  Py_RETURN_NONE;
}

// ---- arguments --------------------------------------------------------------------------------
const at::Tensor* tensor(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

int dtype_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kHalf: return TD_F16;
    case at::kBFloat16: return TD_BF16;
    case at::kFloat: return TD_F32;
    default: return -1;
  }
}
bool dense(const at::Tensor* t) { return t && t->is_cuda() && t->is_contiguous(); }
bool dense(const at::Tensor* t, int dims) { return dense(t) && t->dim() == dims; }
bool i32(const at::Tensor* t) { return t->scalar_type() == at::kInt; }
// two dimensions, dense rows (_check_rows)
bool rows2d(const at::Tensor* t) {
  return t && t->is_cuda() && t->dim() == 2 && (t->numel() == 0 || t->stride(1) == 1);
}
void* ptr(const at::Tensor& t) { return t.data_ptr(); }
template <typename P>
P* ptr_as(const at::Tensor& t) { return reinterpret_cast<P*>(t.data_ptr()); }

bool integer(PyObject* o, int64_t lo, int64_t hi, int64_t& out) {
  if (!PyLong_Check(o)) return false;
  int overflow = 0;
  out = PyLong_AsLongLongAndOverflow(o, &overflow);
  return !overflow && out >= lo && out <= hi;
}
bool number(PyObject* o, double& out) {
  if (PyFloat_CheckExact(o)) {
    out = PyFloat_AS_DOUBLE(o);
    return true;
  }
  int64_t i;
  if (!integer(o, -(1ll << 53), 1ll << 53, i)) return false;
  out = (double)i;
  return true;
}
void* stream_of(PyObject* o) { return PyLong_AsVoidPtr(o); }  // an int from torch

// the KV pool of a layer, as _pool describes it
// (layer >= 0: that of the pools of all layers)
bool pool_of(const at::Tensor* kv, int64_t layout, td_paged_kv& p, int64_t layer = -1) {
  const int at = layer >= 0 ? 1 : 0;  // dimension of the pages
  if (!dense(kv, 5 + at) || kv->size(at + 1) != 2 || (layout != TD_NHD && layout != TD_HND)) return false;
  if (layer >= 0 && layer >= kv->size(0)) return false;
  const int code = dtype_code(*kv);
  if (code < 0) return false;
  p.data = ptr(*kv);
  if (layer > 0) p.data = (char*)p.data + layer * kv->stride(0) * kv->element_size();
  p.max_pages = kv->size(at);
  p.num_kv_heads = (int32_t)kv->size(at + (layout == TD_HND ? 2 : 3));
  p.head_dim = (int32_t)kv->size(at + 4);
  p.page_size = (int32_t)kv->size(at + (layout == TD_HND ? 3 : 2));
  p.layout = (int32_t)layout;
  p.dtype = code;
  return true;
}

PyObject* failed(int rc) {
  const char* msg = lib.last_error();
  if (msg && msg[0])
    PyErr_SetString(PyExc_RuntimeError, msg);
  else
    PyErr_Format(PyExc_RuntimeError, "libtidal_hip call failed with status %d", rc);
  return nullptr;
}

// the library call itself without the interpreter's lock, as ctypes does it: a full launch queue blocks
template <class F, class... A>
int unlocked(F fn, A... args) {  // (what the arguments need the lock for is done before the call)
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = fn(args...);
  Py_END_ALLOW_THREADS
  return rc;
}

struct Names {
  PyObject *begun, *geom, *layout, *workspace, *static_scratch, *chunk_tokens, *waves_per_block, *tile_rows,
      *fused_merge, *sparse_waves, *sparse_rows;
} names;

// a new reference dropped at the end of the scope
struct Ref {
  PyObject* o;
  explicit Ref(PyObject* o) : o(o) {}
  ~Ref() { Py_XDECREF(o); }
  Ref(const Ref&) = delete;
};
bool attr_int(PyObject* self, PyObject* name, int32_t& out) {
  Ref v(PyObject_GetAttr(self, name));
  int64_t x;
  if (!v.o || !integer(v.o, INT32_MIN, INT32_MAX, x)) return false;
  out = (int32_t)x;
  return true;
}

// (self, q, o, paged_kv_data, paged_kv_indices, paged_kv_indptr, last_page_len, last_page_idx, qk_product, slots, lse,
// n_list, fresh, counts, stream).  layer >= 0: paged_kv_data holds the pools of all layers; o null: allocated here
bool forward_layer(PyObject* const* a, int64_t layer, at::Tensor* made, int& rc) {
  PyObject* self = a[0];
  const at::Tensor *q = tensor(a[1]), *o = made ? made : tensor(a[2]), *kv = tensor(a[3]), *idx = tensor(a[4]);
  {
    Ref begun(PyObject_GetAttr(self, names.begun));
    if (begun.o != Py_True) return false;
  }
  int32_t layout;
  td_paged_kv pool;
  if (!attr_int(self, names.layout, layout) || !dense(q, 3) || !rows2d(idx) || !i32(idx) ||
      !pool_of(kv, layout, pool, layer))
    return false;
  if (made) *made = at::empty_like(*q);
  if (!dense(o)) return false;
  int64_t hq, hkv, d, page;
  {
    Ref geom(PyObject_GetAttr(self, names.geom));
    if (!geom.o || !PyTuple_CheckExact(geom.o) || PyTuple_GET_SIZE(geom.o) != 5 ||
        !integer(PyTuple_GET_ITEM(geom.o, 0), 1, INT32_MAX, hq) || !integer(PyTuple_GET_ITEM(geom.o, 1), 1, INT32_MAX, hkv) ||
        !integer(PyTuple_GET_ITEM(geom.o, 2), 1, INT32_MAX, d) || !integer(PyTuple_GET_ITEM(geom.o, 3), 1, INT32_MAX, page) ||
        !THPDtype_Check(PyTuple_GET_ITEM(geom.o, 4)) ||
        reinterpret_cast<THPDtype*>(PyTuple_GET_ITEM(geom.o, 4))->scalar_type != q->scalar_type())
      return false;
  }
  const int64_t batch = q->size(0);
  if (q->size(1) != hq || q->size(2) != d || pool.num_kv_heads != hkv || pool.head_dim != d || pool.page_size != page ||
      kv->scalar_type() != q->scalar_type() || o->scalar_type() != q->scalar_type() || o->sizes() != q->sizes())
    return false;
  const int64_t rows = idx->size(0), budget = idx->size(1);
  if (rows != 1 && rows != hkv && rows != hq) return false;
  const bool slots = a[9] == Py_True;

  td_index_list list = {};
  list.idx = idx->numel() ? ptr_as<int32_t>(*idx) : nullptr;
  list.idx_rows = (int32_t)rows;
  const int64_t row_stride = rows > 1 ? idx->stride(0) : budget;
  if (row_stride < 0 || row_stride > INT32_MAX || budget > INT32_MAX) return false;
  list.idx_row_stride = (int32_t)row_stride;
  list.kind = slots ? TD_IDX_SLOTS : TD_IDX_PAGES;
  if (a[5] != Py_None) {
    const at::Tensor* indptr = tensor(a[5]);
    if (!indptr || !i32(indptr) || indptr->numel() != batch + 1) return false;
    list.indptr = ptr_as<int32_t>(*indptr);
  }
  if (a[13] != Py_None) {
    const at::Tensor* counts = tensor(a[13]);
    if (!counts || !i32(counts) || !list.indptr || counts->numel() != batch) return false;
    list.count_arr = ptr_as<int32_t>(*counts);
  }
  int64_t n_list = budget;
  if (a[11] != Py_None) {
    if (!integer(a[11], INT32_MIN, INT32_MAX, n_list)) return false;
    n_list = n_list < budget ? n_list : budget;
  }
  list.n_list_host = (int32_t)n_list;
  int64_t max_last = page, word;
  if (const at::Tensor* t = tensor(a[6])) {
    if (!i32(t)) return false;
    list.last_page_len_arr = ptr_as<int32_t>(*t);
  } else {
    if (!integer(a[6], INT32_MIN, INT32_MAX, word)) return false;
    list.last_page_len = (int32_t)word;
    max_last = word;
  }
  if (const at::Tensor* t = tensor(a[7])) {
    if (!i32(t)) return false;
    list.last_page_idx_arr = ptr_as<int32_t>(*t);
  } else {
    if (!integer(a[7], INT32_MIN, INT32_MAX, word)) return false;
    list.last_page_idx = (int32_t)word;
  }
  const int64_t max_items = n_list * (slots ? 1 : page) + max_last;

  void* scores = nullptr;
  int scores_dtype = TD_F32;
  int64_t score_stride = 0;
  if (a[8] != Py_None) {
    const at::Tensor* qk = tensor(a[8]);
    if (!qk) return false;
    if (qk->numel() > 0) {
      if (!dense(qk) || qk->numel() % (batch * hq) != 0) return false;
      score_stride = qk->numel() / (batch * hq);
      scores_dtype = dtype_code(*qk);
      if (score_stride < max_items || scores_dtype < 0) return false;
      scores = ptr(*qk);
    }
  }
  float* lse = nullptr;
  if (a[10] != Py_None) {
    const at::Tensor* t = tensor(a[10]);
    if (!dense(t) || t->scalar_type() != at::kFloat || t->numel() != batch * hq) return false;
    lse = ptr_as<float>(*t);
  }
  td_fresh_token fresh, *fresh_arg = nullptr;
  if (a[12] != Py_None) {
    if (!PyTuple_CheckExact(a[12]) || PyTuple_GET_SIZE(a[12]) != 5) return false;
    const at::Tensor* t[5];
    for (int i = 0; i < 5; ++i)
      if (!dense(t[i] = tensor(PyTuple_GET_ITEM(a[12], i)))) return false;
    for (int i = 0; i < 2; ++i)
      if (t[i]->dim() != 3 || t[i]->size(0) != batch || t[i]->size(1) != hkv || t[i]->size(2) != d ||
          t[i]->scalar_type() != q->scalar_type() || t[i + 2]->scalar_type() != at::kFloat ||
          t[i + 2]->numel() != batch * d / 2)
        return false;
    if (!i32(t[4]) || t[4]->numel() != batch) return false;
    fresh = {ptr(*t[0]), ptr(*t[1]), ptr_as<float>(*t[2]), ptr_as<float>(*t[3]), ptr_as<int32_t>(*t[4])};
    fresh_arg = &fresh;
  }

  // the plan is host arithmetic of a fraction of a microsecond: made anew with every call
  td_decode_plan plan = {};
  if (!attr_int(self, names.chunk_tokens, plan.chunk_tokens) || !attr_int(self, names.waves_per_block, plan.waves_per_block) ||
      !attr_int(self, names.tile_rows, plan.tile_rows) || !attr_int(self, names.fused_merge, plan.fused_merge) ||
      !attr_int(self, names.sparse_waves, plan.sparse_waves) || !attr_int(self, names.sparse_rows, plan.sparse_rows))
    return false;
  if (!lib.short_list_pays((int32_t)batch, (int32_t)hq, (int32_t)hkv, (int32_t)d, (int32_t)rows, max_items, list.kind,
                           scores != nullptr))
    plan.sparse_waves = -1;
  if (lib.make_plan((int32_t)batch, (int32_t)hq, (int32_t)hkv, (int32_t)d, (int32_t)rows, max_items, &plan) != TD_OK)
    return false;
  const float scale = (float)(1.0 / std::sqrt((double)d));
  Ref built_in(PyObject_GetAttr(self, names.static_scratch));
  if (built_in.o == Py_True) {
    rc = unlocked(lib.decode_attn_noalloc, &pool, &list, &plan, ptr(*q), ptr(*o), (int32_t)batch, (int32_t)hq, scale,
                  scores, scores_dtype, score_stride, lse, fresh_arg, stream_of(a[14]));
    return true;
  }
  Ref held(PyObject_GetAttr(self, names.workspace));
  const at::Tensor* ws = held.o ? tensor(held.o) : nullptr;
  if (plan.workspace_bytes > 0 && (!ws || ws->numel() < plan.workspace_bytes || ws->device() != q->device())) return false;
  rc = unlocked(lib.decode_attn, &pool, &list, &plan, ptr(*q), ptr(*o), (int32_t)batch, (int32_t)hq, scale, scores,
                scores_dtype, score_stride, lse, fresh_arg, ws ? ptr(*ws) : nullptr, ws ? ws->numel() : 0,
                stream_of(a[14]));
  return true;
}

// BatchDecodeWithPagedKVCachePyTorchWrapper.forward: the arguments of forward_layer
bool forward_regular(PyObject* const* a, int& rc) { return forward_layer(a, -1, nullptr, rc); }

// The same on a layer of the cache's pools (o unused, the layer in front of the stream); the new output
// instead of True.
bool attend_regular(PyObject* const* a, at::Tensor& o, int& rc) {
  int64_t layer;
  return integer(a[15], 0, INT32_MAX, layer) && forward_layer(a, layer, &o, rc);
}

// topk_filtering: (estimated_value, estimated_indices, d_out, indices_out, buf, page_budget, page_table, page_size,
// lengths, upper_bound, segment, stream, columns: None or how many of estimated_value take part)
bool topk_regular(PyObject* const* a, int& rc) {
  const at::Tensor *v = tensor(a[0]), *out = tensor(a[3]);
  int64_t k, page_size;
  if (!rows2d(v) || !rows2d(out) || !i32(out) || !integer(a[5], 0, INT32_MAX, k) || !integer(a[7], 1, INT32_MAX, page_size))
    return false;
  const int code = dtype_code(*v);
  const int64_t rows = v->size(0);
  int64_t len = v->size(1), columns;
  if (a[12] != Py_None) {
    if (!integer(a[12], 0, len, columns)) return false;
    len = columns;
  }
  if (code < 0 || rows < 1 || rows > INT32_MAX || len > INT32_MAX || a[2] != Py_None) return false;
  const int32_t* in_idx = nullptr;
  int64_t in_stride = 0;
  if (a[1] != Py_None) {
    const at::Tensor* t = tensor(a[1]);
    if (!dense(t, 2) || !i32(t) || t->size(0) != rows) return false;
    len = len < t->size(1) ? len : t->size(1);
    in_idx = ptr_as<int32_t>(*t);
    in_stride = t->size(1);
  }
  if (k > len) return false;
  const int32_t *table = nullptr, *lengths = nullptr;
  int64_t table_stride = 0, per = 0;
  if (a[6] != Py_None) {
    const at::Tensor* t = tensor(a[6]);
    if (!dense(t) || !i32(t)) return false;
    if (t->dim() == 2) {
      const int64_t groups = t->size(0);
      if (groups < 1 || rows % groups) return false;
      table_stride = t->stride(0);
      per = rows / groups;
    } else if (t->dim() != 1) {
      return false;
    }
    if (t->size(-1) * page_size < len) return false;
    table = ptr_as<int32_t>(*t);
  }
  if (a[8] != Py_None) {
    const at::Tensor* t = tensor(a[8]);
    if (!dense(t) || !i32(t)) return false;
    const int64_t groups = t->numel();
    if (groups < 1 || rows % groups || (per && per != rows / groups)) return false;
    per = rows / groups;
    lengths = ptr_as<int32_t>(*t);
  }
  int64_t group_stride = 0;
  if (a[10] == Py_None) {
    if (out->size(0) != rows || out->size(1) != k) return false;
  } else {
    int64_t segment;
    const int64_t in_group = per ? per : rows;
    if (!integer(a[10], 1, INT32_MAX, segment) || segment < k || out->size(0) != in_group ||
        out->size(1) < rows / in_group * segment)
      return false;
    group_stride = segment;
  }
  const float* bound = nullptr;
  if (a[9] != Py_None) {
    const at::Tensor* t = tensor(a[9]);
    if (!dense(t) || t->scalar_type() != at::kFloat || t->numel() != rows) return false;
    bound = ptr_as<float>(*t);
  }
  void* ws = nullptr;
  int64_t ws_bytes = 0;
  if (const at::Tensor* t = tensor(a[4])) {
    if (dense(t) && (int64_t)(t->numel() * t->element_size()) >= lib.topk_workspace_bytes((int32_t)rows)) {
      ws = ptr(*t);
      ws_bytes = t->numel() * t->element_size();
    }
  }
  rc = unlocked(lib.topk_segments, ptr(*v), code, v->stride(0), (int32_t)rows, (int32_t)len, (int32_t)k, in_idx,
                in_stride, table, table_stride, (int32_t)per, lengths, (int32_t)page_size, bound, nullptr,
                ptr_as<int32_t>(*out), out->stride(0), group_stride, ws, ws_bytes, stream_of(a[11]));
  return true;
}

// rope_table: (positions, head_dim, rope_scale, rope_theta, stream), cos and sin allocated here
bool rope_table_regular(PyObject* const* a, at::Tensor& cos, at::Tensor& sin, int& rc) {
  const at::Tensor* pos = tensor(a[0]);
  int64_t d;
  double scale, theta;
  if (!dense(pos) || !i32(pos) || !integer(a[1], 2, INT32_MAX, d) || !number(a[2], scale) || !number(a[3], theta))
    return false;
  const auto options = pos->options().dtype(at::kFloat);
  cos = at::empty({pos->numel(), d / 2}, options);
  sin = at::empty({pos->numel(), d / 2}, options);
  rc = unlocked(lib.rope_table, ptr_as<int32_t>(*pos), (int32_t)pos->numel(), (int32_t)d, (float)scale, (float)theta,
                ptr_as<float>(cos), ptr_as<float>(sin), stream_of(a[4]));
  return true;
}

// apply_rope_in_place: (q, k, past_kv_len, rope_scale, rope_theta, stream)
bool rope_in_place_regular(PyObject* const* a, int& rc) {
  const at::Tensor *q = tensor(a[0]), *k = tensor(a[1]);
  int64_t past;
  double scale, theta;
  if (!dense(q, 3) || !dense(k, 3) || q->size(0) != k->size(0) || q->size(2) != k->size(2) ||
      q->scalar_type() != k->scalar_type() || !integer(a[2], INT64_MIN, INT64_MAX, past) || !number(a[3], scale) ||
      !number(a[4], theta))
    return false;
  const int code = dtype_code(*q);
  if (code < 0) return false;
  rc = unlocked(lib.rope_in_place, ptr(*q), ptr(*k), (int32_t)q->size(0), (int32_t)q->size(1), (int32_t)k->size(1),
                (int32_t)q->size(2), past, (float)scale, (float)theta, code, stream_of(a[5]));
  return true;
}

// _append: (k, v, kv_data, kv_indices, kv_indptr, kv_last_page_len, metadata_data, metadata_indices, metadata_indptr,
// metadata_last_page_len, layout, decode, stream, layer: that of kv_data's pools of all layers, or -1)
bool append_regular(PyObject* const* a, int& rc) {
  const at::Tensor *k = tensor(a[0]), *v = tensor(a[1]), *kv = tensor(a[2]), *idx = tensor(a[3]), *indptr = tensor(a[4]);
  int64_t last, layout, layer, meta_last = 0;
  td_paged_kv pool, meta_pool, *meta = nullptr;
  if (!dense(k, 3) || !dense(v, 3) || !dense(idx, 1) || !i32(idx) || !indptr || !i32(indptr) ||
      !integer(a[5], INT32_MIN, INT32_MAX, last) || !integer(a[10], 0, 1, layout) ||
      !integer(a[13], -1, INT32_MAX, layer) || !pool_of(kv, layout, pool, layer))
    return false;
  if ((a[11] == Py_True && k->size(0) != 1) || k->sizes() != v->sizes() || k->scalar_type() != v->scalar_type() ||
      pool.num_kv_heads != k->size(1) || pool.head_dim != k->size(2) || kv->scalar_type() != k->scalar_type())
    return false;
  const int32_t *meta_idx = nullptr, *meta_indptr = nullptr;
  if (a[6] != Py_None) {
    const at::Tensor *m = tensor(a[6]), *mi = tensor(a[7]), *mp = tensor(a[8]);
    if (!m || m->numel() == 0 || !pool_of(m, layout, meta_pool) || !dense(mi, 1) || !i32(mi) || mi->numel() == 0 ||
        !mp || !i32(mp) || mp->numel() == 0 || !integer(a[9], INT32_MIN, INT32_MAX, meta_last))
      return false;
    meta = &meta_pool;
    meta_idx = ptr_as<int32_t>(*mi);
    meta_indptr = ptr_as<int32_t>(*mp);
  }
  rc = unlocked(lib.append_kv, &pool, ptr(*k), ptr(*v), (int32_t)k->size(0), ptr_as<int32_t>(*idx),
                ptr_as<int32_t>(*indptr), (int32_t)last, meta, meta_idx, meta_indptr, (int32_t)meta_last,
                stream_of(a[12]));
  return true;
}

// prefill_with_paged_kv_cache: (q, kv_data, kv_indices, kv_last_page_len, causal, layout, stream, layer: that of
// kv_data's pools of all layers, or -1); the output and the scratch of this call alone are allocated here
bool prefill_regular(PyObject* const* a, at::Tensor& o, int& rc) {
  const at::Tensor *q = tensor(a[0]), *kv = tensor(a[1]), *idx = tensor(a[2]);
  int64_t last, layout, layer;
  td_paged_kv pool;
  if (!dense(q, 3) || !dense(idx) || !i32(idx) || !integer(a[3], INT32_MIN, INT32_MAX, last) || !PyBool_Check(a[4]) ||
      !integer(a[5], 0, 1, layout) || !integer(a[7], -1, INT32_MAX, layer) || !pool_of(kv, layout, pool, layer))
    return false;
  const int64_t n_pages = idx->numel(), kv_len = (n_pages - 1) * pool.page_size + last;
  const int causal = a[4] == Py_True;
  if (q->size(2) != pool.head_dim || q->scalar_type() != kv->scalar_type() || kv_len < 0 || kv_len > INT32_MAX) return false;
  o = at::empty_like(*q);
  int64_t bytes = lib.prefill_workspace_bytes(&pool, (int32_t)kv_len, (int32_t)q->size(0), (int32_t)q->size(1), causal);
  at::Tensor scratch;  // (torch's allocator hands it out again in stream order)
  if (bytes > 0) {
    try {
      scratch = at::empty({bytes}, q->options().dtype(at::kByte));
    } catch (const c10::OutOfMemoryError&) {  // slower without, but a call needs none
      bytes = 0;
    }
  }
  rc = unlocked(lib.prefill_attn_split, &pool, ptr_as<int32_t>(*idx), (int32_t)n_pages, (int32_t)kv_len, ptr(*q),
                ptr(o), (int32_t)q->size(0), (int32_t)q->size(1), (float)(1.0 / std::sqrt((double)pool.head_dim)),
                causal, bytes > 0 ? ptr(scratch) : nullptr, bytes, stream_of(a[6]));
  return true;
}

// gemv: (weight, x, norm_weight, eps, gated, residual, pair_gated, out, stream)
bool gemv_regular(PyObject* const* a, int& rc) {
  const at::Tensor *w = tensor(a[0]), *x = tensor(a[1]), *out = tensor(a[7]);
  double eps;
  if (!w || !w->is_cuda() || w->dim() != 2 || w->stride(1) != 1 || !dense(x) || !dense(out) || !number(a[3], eps)) return false;
  const int64_t rows = w->size(0), cols = w->size(1);
  const bool gated = a[4] == Py_True, pair = a[6] == Py_True;
  const int code = dtype_code(*w);
  if (code < 0 || rows > INT32_MAX || cols > INT32_MAX || w->scalar_type() != x->scalar_type() ||
      x->numel() != (gated ? 2 * cols : cols) || out->scalar_type() != x->scalar_type() ||
      out->numel() != (pair ? rows / 2 : rows) || (pair && (rows % 2 || gated || a[5] != Py_None)))
    return false;
  const void *norm = nullptr, *residual = nullptr;
  if (a[2] != Py_None) {
    const at::Tensor* t = tensor(a[2]);
    if (gated || !dense(t) || t->numel() != cols || t->scalar_type() != x->scalar_type()) return false;
    norm = ptr(*t);
  }
  if (a[5] != Py_None) {
    const at::Tensor* t = tensor(a[5]);
    if (!dense(t) || t->numel() != rows || t->scalar_type() != x->scalar_type()) return false;
    residual = ptr(*t);
  }
  rc = unlocked(lib.gemv, ptr(*w), w->stride(0), (int32_t)rows, (int32_t)cols, ptr(*x), norm ? 1 : (gated ? 2 : 0),
                norm, (float)eps, residual, pair ? 1 : 0, ptr(*out), code, stream_of(a[8]));
  return true;
}

// score_reduce: (logits, lse, num_kv_heads, n, mode, out, stream)
bool score_reduce_regular(PyObject* const* a, int& rc) {
  const at::Tensor *logits = tensor(a[0]), *lse = tensor(a[1]), *out = tensor(a[5]);
  int64_t hkv, n, mode;
  if (!dense(logits, 2) || !dense(lse) || logits->scalar_type() != at::kFloat || lse->scalar_type() != at::kFloat ||
      lse->numel() != logits->size(0) || !out || out->dim() != 2 || !integer(a[2], 1, INT32_MAX, hkv) ||
      !integer(a[3], 0, INT32_MAX, n) || !integer(a[4], 0, 1, mode))
    return false;
  rc = unlocked(lib.score_reduce, ptr_as<float>(*logits), logits->stride(0), ptr_as<float>(*lse),
                (int32_t)logits->size(0), (int32_t)hkv, (int32_t)n, (int32_t)mode, ptr_as<float>(*out),
                out->stride(0), stream_of(a[6]));
  return true;
}

// estimate_attn_score: (q, o, metadata_data, metadata_indices, metadata_last_page_len, layout, stream)
bool estimate_regular(PyObject* const* a, int& rc) {
  const at::Tensor *q = tensor(a[0]), *o = tensor(a[1]), *meta = tensor(a[2]), *idx = tensor(a[3]);
  int64_t last, layout;
  td_paged_kv pool;
  if (!dense(q, 3) || !dense(o, 2) || !dense(idx) || !i32(idx) || !integer(a[4], INT32_MIN, INT32_MAX, last) ||
      !integer(a[5], 0, 1, layout) || !pool_of(meta, layout, pool))
    return false;
  const int64_t n_pages = idx->numel();
  if (q->size(0) != 1 || q->size(2) != pool.head_dim || q->scalar_type() != meta->scalar_type() ||
      o->scalar_type() != q->scalar_type() || o->size(0) != q->size(1) ||
      o->size(1) < (n_pages - 1) * pool.page_size + last - 1)
    return false;
  rc = unlocked(lib.estimate_score, &pool, ptr_as<int32_t>(*idx), (int32_t)n_pages, (int32_t)last, ptr(*q),
                (int32_t)q->size(1), ptr(*o), o->stride(0), stream_of(a[6]));
  return true;
}

// run(rc) and its outcome: False, an exception, or what result() makes of a launch
template <class Run, class Result>
PyObject* outcome(Run run, Result result) {
  int rc = TD_OK;
  try {
    if (!run(rc)) {
      PyErr_Clear();
      Py_RETURN_FALSE;
    }
  } catch (const std::exception&) {  // a tensor without storage and the like: Python says what is wrong
    PyErr_Clear();
    Py_RETURN_FALSE;
  }
  if (PyErr_Occurred()) return nullptr;
  return rc == TD_OK ? result() : failed(rc);
}
bool takes(Py_ssize_t n, Py_ssize_t wanted) {
  if (n != wanted) PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", wanted, n);
  return n == wanted;
}

template <bool (*F)(PyObject* const*, int&), int N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!takes(n, N)) return nullptr;
  return outcome([&](int& rc) { return F(args, rc); }, [] { Py_RETURN_TRUE; });
}
template <bool (*F)(PyObject* const*, at::Tensor&, int&), int N>
PyObject* maker(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!takes(n, N)) return nullptr;
  at::Tensor o;
  return outcome([&](int& rc) { return F(args, o, rc); }, [&] { return THPVariable_Wrap(std::move(o)); });
}
PyObject* rope_table(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!takes(n, 5)) return nullptr;
  at::Tensor cos, sin;
  return outcome([&](int& rc) { return rope_table_regular(args, cos, sin, rc); },
                 [&]() -> PyObject* {
                   PyObject* pair = PyTuple_New(2);
                   if (!pair) return nullptr;
                   PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(std::move(cos)));
                   PyTuple_SET_ITEM(pair, 1, THPVariable_Wrap(std::move(sin)));
                   return pair;
                 });
}

#define TD_ENTRY(name, fn, n) {name, (PyCFunction)(void (*)(void))(entry<fn, n>), METH_FASTCALL, nullptr}
#define TD_MAKER(name, fn, n) {name, (PyCFunction)(void (*)(void))(maker<fn, n>), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"bind", bind, METH_O, "addresses of libtidal_hip.so's entry points by name"},
    TD_ENTRY("forward", forward_regular, 15),
    TD_ENTRY("topk", topk_regular, 13),
    TD_MAKER("attend", attend_regular, 16),
    {"rope_table", (PyCFunction)(void (*)(void))rope_table, METH_FASTCALL, nullptr},
    TD_ENTRY("rope_in_place", rope_in_place_regular, 6),
    TD_ENTRY("append", append_regular, 14),
    TD_MAKER("prefill", prefill_regular, 8),
    TD_ENTRY("gemv", gemv_regular, 9),
    TD_ENTRY("score_reduce", score_reduce_regular, 7),
    TD_ENTRY("estimate", estimate_regular, 7),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host_calls(void) {
  struct { PyObject** at; const char* name; } interned[] = {
      {&names.begun, "_begun"}, {&names.geom, "_geom"}, {&names.layout, "_layout"}, {&names.workspace, "_workspace"},
      {&names.static_scratch, "static_scratch"}, {&names.chunk_tokens, "chunk_tokens"},
      {&names.waves_per_block, "waves_per_block"}, {&names.tile_rows, "tile_rows"}, {&names.fused_merge, "fused_merge"},
      {&names.sparse_waves, "sparse_waves"}, {&names.sparse_rows, "sparse_rows"}};
  for (auto& n : interned)
    if (!(*n.at = PyUnicode_InternFromString(n.name))) return nullptr;
  return PyModule_Create(&module);
}
