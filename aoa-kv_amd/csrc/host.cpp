// aoakv._host: the torch-tensor wrappers of the entry points on the decode and
// prefill paths (aoakv/ops.py), in C++.
//
// A call here checks dtypes, devices and shapes as the Python wrappers of the
// other entry points do, with the same exceptions, and calls the C ABI with
// raw device pointers on torch's current stream.  The checks of one call's 12
// or so tensors, the current stream and a ctypes call of 20 arguments took
// 10 to 15 us in Python, more than the kernels of a short decode step; here
// about 2 us (a token's RoPE and append, called back to back, went from 18.8 to
// 5.7 us; estimate, top-k and attention at 4096 tokens from 36.6 to 18.9).
// The library itself is the one aoakv._lib loaded (bind), and a non-zero
// status raises its AoakvError.
#include <Python.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/autograd/python_variable.h>

#include <exception>
#include <sstream>
#include <string>
#include <type_traits>

#include "../../include/aoakv.h"

namespace {

using at::Tensor;

// A Python exception that is already set.
struct PyErr {};

#define FOR_EACH_ENTRY(X)                                                              \
  X(append_kv_cache_prefill) X(append_kv_cache_decode) X(rope_append_kv_cache_decode)  \
  X(rope_append_kv_cache_prefill) X(rms_norm_forward) X(estimate_attn_score)           \
  X(topk_filtering) X(decode_sparse_attn) X(sparse_decode_layer)                       \
  X(prefill_workspace_size) X(prefill_with_workspace) X(last_error)

struct Lib {
#define X(n) decltype(&aoakv_##n) n = nullptr;
  FOR_EACH_ENTRY(X)
#undef X
} g_lib;
PyObject* g_error = nullptr;      // aoakv._lib.AoakvError
PyObject* g_arg_error = nullptr;  // ctypes.ArgumentError

[[noreturn]] void raise(PyObject* type, const std::string& msg) {
  PyErr_SetString(type, msg.c_str());
  throw PyErr{};
}

std::string shape_str(const Tensor& t) {
  std::ostringstream s;
  s << '(';
  for (int64_t i = 0; i < t.dim(); ++i) s << (i ? ", " : "") << t.size(i);
  s << (t.dim() == 1 ? ",)" : ")");
  return s.str();
}

const char* dtype_name(at::ScalarType t) {
  return t == at::kHalf ? "torch.float16" : t == at::kFloat ? "torch.float32"
         : t == at::kInt ? "torch.int32" : "torch.uint8";
}

// A contiguous device tensor of this dtype.
const Tensor& need(PyObject* o, const char* name, at::ScalarType dtype) {
  if (!THPVariable_Check(o)) raise(PyExc_TypeError, std::string(name) + " must be a torch.Tensor");
  const Tensor& t = THPVariable_Unpack(o);
  if (t.scalar_type() != dtype) {
    PyObject* d = PyObject_GetAttrString(o, "dtype");
    PyErr_Format(PyExc_TypeError, "%s must be %s, got %S", name, dtype_name(dtype), d);
    Py_XDECREF(d);
    throw PyErr{};
  }
  if (!t.is_cuda()) raise(PyExc_ValueError, std::string(name) + " must be a device tensor");
  if (!t.is_contiguous()) raise(PyExc_ValueError, std::string(name) + " must be contiguous");
  return t;
}
const Tensor& f16(PyObject* o, const char* name) { return need(o, name, at::kHalf); }
const int32_t* i32(PyObject* o, const char* name) {
  return static_cast<const int32_t*>(need(o, name, at::kInt).data_ptr());
}
const int32_t* i32_or_null(PyObject* o, const char* name) {
  return o == Py_None ? nullptr : i32(o, name);
}
void* ptr(const Tensor& t) { return t.data_ptr(); }
// the address of any tensor (the fused layer takes its page tables unchecked)
void* any_ptr(PyObject* o, const char* name) {
  if (!THPVariable_Check(o))
    raise(PyExc_AttributeError, std::string(name) + " must be a torch.Tensor");
  return THPVariable_Unpack(o).data_ptr();
}
const int32_t* table(PyObject* o) {
  return static_cast<const int32_t*>(any_ptr(o, "a page table"));
}
// v_log_norm: checked where the flags use it
const void* log_norm_or_null(PyObject* o, uint32_t flags) {
  if (flags & AOAKV_FLAG_VALUE_AWARE) return ptr(f16(o, "v_log_norm"));
  return o == Py_None ? nullptr : any_ptr(o, "v_log_norm");
}

// An unsigned 32-bit argument: a Python int, as ctypes takes it.
uint32_t u32(PyObject* o) {
  if (!PyLong_Check(o)) raise(g_arg_error, "int expected");
  const unsigned long v = PyLong_AsUnsignedLongMask(o);
  if (v == (unsigned long)-1 && PyErr_Occurred()) throw PyErr{};
  return (uint32_t)v;
}
// ... that is no more than a size: the whole number is compared
uint32_t u32_at_most(PyObject* o, int64_t size, const char* msg) {
  const uint32_t v = u32(o);
  int big = 0;
  const long long x = PyLong_AsLongLongAndOverflow(o, &big);
  if (big != 0 || x < 0 || x > size) raise(PyExc_ValueError, msg);
  return v;
}
// o == n, as Python compares them
bool equals(PyObject* o, unsigned long n) {
  PyObject* x = PyLong_FromUnsignedLong(n);
  const int r = x == nullptr ? -1 : PyObject_RichCompareBool(o, x, Py_EQ);
  Py_XDECREF(x);
  if (r < 0) throw PyErr{};
  return r != 0;
}
float f32(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw PyErr{};
  return (float)v;
}

struct Dims {
  uint32_t S, H, D, layout;
};
// [max_pages, 2, S, H, D] (NHD) or [max_pages, 2, H, S, D] (HND)
Dims cache_dims(const Tensor& kv, PyObject* layout) {
  if (kv.dim() != 5 || kv.size(1) != 2)
    raise(PyExc_ValueError, "paged cache must be 5-d [pages, 2, ., ., D], got " + shape_str(kv));
  int big = 0;
  const long x = PyLong_Check(layout) ? PyLong_AsLongAndOverflow(layout, &big) : -1;
  if (x != (long)AOAKV_LAYOUT_NHD && x != (long)AOAKV_LAYOUT_HND &&
      !equals(layout, AOAKV_LAYOUT_NHD) && !equals(layout, AOAKV_LAYOUT_HND)) {
    PyErr_Format(PyExc_ValueError, "unknown layout %S", layout);
    throw PyErr{};
  }
  const uint32_t l = u32(layout);
  const bool nhd = l == AOAKV_LAYOUT_NHD;
  return Dims{(uint32_t)kv.size(nhd ? 2 : 3), (uint32_t)kv.size(nhd ? 3 : 2),
              (uint32_t)kv.size(4), l};
}
bool is_shape(const Tensor& t, int64_t a, int64_t b, int64_t c) {
  return t.dim() == 3 && t.size(0) == a && t.size(1) == b && t.size(2) == c;
}

void* stream() { return c10::hip::getCurrentHIPStream().stream(); }

// The interpreter lock given up for a scope (taken again on an exception too).
struct Unlocked {
  PyThreadState* s = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(s); }
};

// Calls an entry point without the interpreter lock; raises on its status.
template <class F>
void call(const char* name, F&& f) {
  int rc;
  {
    Unlocked u;
    rc = f();
  }
  if (rc == AOAKV_OK) return;
  PyObject* e = PyObject_CallFunction(g_error, "sis", name, rc, g_lib.last_error());
  if (e != nullptr) {
    PyErr_SetObject(g_error, e);
    Py_DECREF(e);
  }
  throw PyErr{};
}

// the cache's tensors of the append calls
struct Cache {
  const Tensor *kv, *meta, *log_norm, *mean;
};
Cache cache_args(PyObject* kv, PyObject* meta, PyObject* log_norm, PyObject* mean) {
  return Cache{&f16(kv, "kv_data"), &f16(meta, "metadata_data"), &f16(log_norm, "v_log_norm"),
               &f16(mean, "v_mean")};
}

// (k, v, kv_data, kv_indices, num_kv_pages, kv_last_page_len, metadata_data,
//  metadata_indices, v_log_norm, v_mean, layout)
void append_kv_cache_prefill(PyObject* const* a) {
  const Tensor &k = f16(a[0], "k"), &v = f16(a[1], "v");
  const Cache c = cache_args(a[2], a[6], a[8], a[9]);
  const int32_t *idx = i32(a[3], "kv_indices"), *midx = i32(a[7], "metadata_indices");
  const Dims d = cache_dims(*c.kv, a[10]);
  const int64_t N = k.dim() == 3 ? k.size(0) : 0;
  if (!is_shape(k, N, d.H, d.D) || !is_shape(v, N, d.H, d.D))
    raise(PyExc_ValueError, "k/v must be [N, " + std::to_string(d.H) + ", " +
                                std::to_string(d.D) + "], got " + shape_str(k) + " / " +
                                shape_str(v));
  const uint32_t pages = u32_at_most(a[4], THPVariable_Unpack(a[3]).numel(),
                                     "kv_indices shorter than num_kv_pages"),
                 last = u32(a[5]);
  void* s = stream();
  call("aoakv_append_kv_cache_prefill", [&] {
    return g_lib.append_kv_cache_prefill(ptr(k), ptr(v), (uint32_t)N, ptr(*c.kv), idx, pages,
                                         last, ptr(*c.meta), midx, ptr(*c.log_norm),
                                         ptr(*c.mean), d.H, d.D, d.S, d.layout, s);
  });
}

// (q, k, v, kv_data, kv_indices, num_kv_pages, kv_last_page_len,
//  metadata_data, metadata_indices, v_log_norm, v_mean, layout, rope_scale,
//  rope_theta)
void rope_append_kv_cache_prefill(PyObject* const* a) {
  const Tensor &q = f16(a[0], "q"), &k = f16(a[1], "k"), &v = f16(a[2], "v");
  const Cache c = cache_args(a[3], a[7], a[9], a[10]);
  const int32_t *idx = i32(a[4], "kv_indices"), *midx = i32(a[8], "metadata_indices");
  const Dims d = cache_dims(*c.kv, a[11]);
  const int64_t N = k.dim() == 3 ? k.size(0) : 0;
  if (!is_shape(k, N, d.H, d.D) || !is_shape(v, N, d.H, d.D))
    raise(PyExc_ValueError, "k/v must be [N, " + std::to_string(d.H) + ", " +
                                std::to_string(d.D) + "], got " + shape_str(k) + " / " +
                                shape_str(v));
  if (q.dim() != 3 || q.size(0) != N || q.size(2) != d.D)
    raise(PyExc_ValueError, "q must be [" + std::to_string(N) + ", Hq, " + std::to_string(d.D) +
                                "], got " + shape_str(q));
  const uint32_t pages = u32_at_most(a[5], THPVariable_Unpack(a[4]).numel(),
                                     "kv_indices shorter than num_kv_pages"),
                 last = u32(a[6]);
  const float scale = f32(a[12]), theta = f32(a[13]);
  void* s = stream();
  call("aoakv_rope_append_kv_cache_prefill", [&] {
    return g_lib.rope_append_kv_cache_prefill(
        ptr(q), ptr(k), ptr(v), (uint32_t)N, (uint32_t)q.size(1), ptr(*c.kv), idx, pages, last,
        ptr(*c.meta), midx, ptr(*c.log_norm), ptr(*c.mean), d.H, d.D, d.S, d.layout, scale, theta,
        s);
  });
}

struct Tables {
  const int32_t *indptr, *indices, *last, *m_indptr, *m_indices;
};
// kv_indptr, kv_indices, kv_last_page_len, metadata_indptr, metadata_indices
// of a batch of B sequences
Tables append_tables(PyObject* const* t, PyObject* const* m, int64_t B) {
  const Tables r{i32(t[0], "kv_indptr"), i32(t[1], "kv_indices"), i32(t[2], "kv_last_page_len"),
                 i32(m[0], "metadata_indptr"), i32(m[1], "metadata_indices")};
  if (THPVariable_Unpack(t[0]).numel() != B + 1 || THPVariable_Unpack(t[2]).numel() != B ||
      THPVariable_Unpack(m[0]).numel() != B + 1)
    raise(PyExc_ValueError, "indptr / last_page_len sizes do not match the batch");
  return r;
}

// (k, v, kv_data, kv_indptr, kv_indices, kv_last_page_len, metadata_data,
//  metadata_indptr, metadata_indices, v_log_norm, v_mean, layout)
void append_kv_cache_decode(PyObject* const* a) {
  const Tensor &k = f16(a[0], "k"), &v = f16(a[1], "v");
  const Cache c = cache_args(a[2], a[6], a[9], a[10]);
  const Dims d = cache_dims(*c.kv, a[11]);
  const int64_t B = k.dim() ? k.size(0) : 0;
  if (!is_shape(k, B, d.H, d.D) || !is_shape(v, B, d.H, d.D))
    raise(PyExc_ValueError,
          "k/v must be [B, " + std::to_string(d.H) + ", " + std::to_string(d.D) + "]");
  const Tables t = append_tables(a + 3, a + 7, B);
  void* s = stream();
  call("aoakv_append_kv_cache_decode", [&] {
    return g_lib.append_kv_cache_decode(ptr(k), ptr(v), (uint32_t)B, ptr(*c.kv), t.indptr,
                                        t.indices, t.last, ptr(*c.meta), t.m_indptr, t.m_indices,
                                        ptr(*c.log_norm), ptr(*c.mean), d.H, d.D, d.S, d.layout,
                                        s);
  });
}

// (q, k, v, kv_data, kv_indptr, kv_indices, kv_last_page_len, metadata_data,
//  metadata_indptr, metadata_indices, v_log_norm, v_mean, layout, rope_scale,
//  rope_theta)
void rope_append_kv_cache_decode(PyObject* const* a) {
  const Tensor &q = f16(a[0], "q"), &k = f16(a[1], "k"), &v = f16(a[2], "v");
  const Cache c = cache_args(a[3], a[7], a[10], a[11]);
  const Dims d = cache_dims(*c.kv, a[12]);
  const int64_t B = k.dim() ? k.size(0) : 0;
  if (!is_shape(k, B, d.H, d.D) || !is_shape(v, B, d.H, d.D) || q.dim() != 3 ||
      q.size(0) != B || q.size(2) != d.D)
    raise(PyExc_ValueError, "q must be [B, Hq, " + std::to_string(d.D) + "], k/v [B, " +
                                std::to_string(d.H) + ", " + std::to_string(d.D) + "]");
  const Tables t = append_tables(a + 4, a + 8, B);
  const float scale = f32(a[13]), theta = f32(a[14]);
  void* s = stream();
  call("aoakv_rope_append_kv_cache_decode", [&] {
    return g_lib.rope_append_kv_cache_decode(
        ptr(q), ptr(k), ptr(v), (uint32_t)B, (uint32_t)q.size(1), ptr(*c.kv), t.indptr, t.indices,
        t.last, ptr(*c.meta), t.m_indptr, t.m_indices, ptr(*c.log_norm), ptr(*c.mean), d.H, d.D,
        d.S, d.layout, scale, theta, s);
  });
}

// (q, scores, metadata_data, metadata_indptr, metadata_indices, kv_indptr,
//  kv_indices, kv_last_page_len, v_log_norm, max_pages, layout, flags)
void estimate_attn_score(PyObject* const* a) {
  const Tensor &q = f16(a[0], "q"), &scores = need(a[1], "scores", at::kFloat),
               &meta = f16(a[2], "metadata_data");
  const int32_t *mip = i32(a[3], "metadata_indptr"), *mix = i32(a[4], "metadata_indices"),
                *ip = i32(a[5], "kv_indptr"), *ix = i32(a[6], "kv_indices"),
                *lpl = i32(a[7], "kv_last_page_len");
  const uint32_t max_pages = u32(a[9]), flags = u32(a[11]);
  const void* log_norm = log_norm_or_null(a[8], flags);
  const Dims d = cache_dims(meta, a[10]);
  if (q.dim() != 3) raise(PyExc_ValueError, "q must be [B, Hq, D], got " + shape_str(q));
  if (q.size(2) != d.D || scores.dim() != 3 || scores.size(0) != q.size(0) ||
      scores.size(1) != d.H)
    raise(PyExc_ValueError, "scores must be [B, " + std::to_string(d.H) + ", >= max_pages]");
  void* s = stream();
  call("aoakv_estimate_attn_score", [&] {
    return g_lib.estimate_attn_score(ptr(q), static_cast<float*>(ptr(scores)),
                                     (uint32_t)scores.size(2), ptr(meta), mip, mix, ip, ix, lpl,
                                     log_norm, (uint32_t)q.size(0), max_pages,
                                     (uint32_t)q.size(1), d.H, d.D, d.S, d.layout, flags, s);
  });
}

// (scores, kv_indptr, kv_indices, kv_last_page_len, token_budget, sel_pages,
//  page_size, flags, token_budgets, workspace)
void topk_filtering(PyObject* const* a) {
  const Tensor &scores = need(a[0], "scores", at::kFloat), &sel = need(a[5], "sel_pages", at::kInt);
  const int32_t *ip = i32(a[1], "kv_indptr"), *ix = i32(a[2], "kv_indices"),
                *lpl = i32(a[3], "kv_last_page_len"),
                *budgets = i32_or_null(a[8], "token_budgets");
  if (scores.dim() != 3)
    raise(PyExc_ValueError, "scores must be [B, Hkv, stride], got " + shape_str(scores));
  if (sel.dim() != 3 || sel.size(0) != scores.size(0) || sel.size(1) != scores.size(1))
    raise(PyExc_ValueError, "sel_pages must be [B, Hkv, k_max]");
  uint32_t* err = nullptr;
  if (a[9] != Py_None) {
    const Tensor& ws = need(a[9], "workspace", at::kByte);
    if (ws.numel() < 12) raise(PyExc_ValueError, "workspace too small to hold the error word");
    err = static_cast<uint32_t*>(ptr(ws)) + AOAKV_WS_ERR_WORD;
  }
  const uint32_t budget = u32(a[4]), page = u32(a[6]), flags = u32(a[7]);
  void* s = stream();
  call("aoakv_topk_filtering", [&] {
    return g_lib.topk_filtering(static_cast<const float*>(ptr(scores)), (uint32_t)scores.size(2),
                                ip, ix, lpl, budget, budgets, static_cast<int32_t*>(ptr(sel)),
                                (uint32_t)sel.size(2), (uint32_t)scores.size(0),
                                (uint32_t)scores.size(1), page, flags, err, s);
  });
}

// (q, o, kv_data, kv_indptr, kv_indices, kv_last_page_len, sel_pages,
//  token_budget, workspace, max_pages, num_kv_heads, layout, token_budgets,
//  flags)
void decode_sparse_attn(PyObject* const* a) {
  const Tensor &q = f16(a[0], "q"), &o = f16(a[1], "o"), &kv = f16(a[2], "kv_data"),
               &ws = need(a[8], "workspace", at::kByte);
  const int32_t *ip = i32(a[3], "kv_indptr"), *ix = i32(a[4], "kv_indices"),
                *lpl = i32(a[5], "kv_last_page_len"), *sel = i32_or_null(a[6], "sel_pages"),
                *budgets = i32_or_null(a[12], "token_budgets");
  const Dims d = cache_dims(kv, a[11]);
  if (!equals(a[10], d.H)) raise(PyExc_ValueError, "num_kv_heads does not match kv_data");
  if (q.dim() != 3) raise(PyExc_ValueError, "q must be [B, Hq, D], got " + shape_str(q));
  if (q.sizes() != o.sizes()) raise(PyExc_ValueError, "o must have q's shape");
  uint32_t sel_stride = 0u;
  if (sel != nullptr || a[6] != Py_None) {
    const Tensor& t = THPVariable_Unpack(a[6]);
    sel_stride = t.dim() ? (uint32_t)t.size(-1) : 0u;
  }
  const uint32_t budget = u32(a[7]), max_pages = u32(a[9]), flags = u32(a[13]);
  void* s = stream();
  call("aoakv_decode_sparse_attn", [&] {
    return g_lib.decode_sparse_attn(ptr(q), ptr(o), ptr(kv), ip, ix, lpl, sel, sel_stride, budget,
                                    budgets, ptr(ws), (size_t)ws.numel(), (uint32_t)q.size(0),
                                    max_pages, (uint32_t)q.size(1), d.H, d.D, d.S, d.layout,
                                    flags, s);
  });
}

// (q, o, kv_data, kv_indptr, kv_indices, kv_last_page_len, metadata_data,
//  metadata_indptr, metadata_indices, v_log_norm, scores, sel_pages,
//  token_budget, workspace, max_pages, layout, flags, token_budgets)
void sparse_decode_layer(PyObject* const* a) {
  const Tensor &q = f16(a[0], "q"), &o = f16(a[1], "o"), &kv = f16(a[2], "kv_data"),
               &meta = f16(a[6], "metadata_data"), &scores = need(a[10], "scores", at::kFloat),
               &sel = need(a[11], "sel_pages", at::kInt), &ws = need(a[13], "workspace", at::kByte);
  const uint32_t flags = u32(a[16]);
  const void* log_norm = log_norm_or_null(a[9], flags);
  const int32_t *budgets = i32_or_null(a[17], "token_budgets"), *ip = table(a[3]),
                *ix = table(a[4]), *lpl = table(a[5]), *mip = table(a[7]), *mix = table(a[8]);
  const Dims d = cache_dims(kv, a[15]);
  if (q.dim() != 3) raise(PyExc_ValueError, "q must be [B, Hq, D], got " + shape_str(q));
  if (scores.dim() == 0 || sel.dim() == 0)
    raise(PyExc_ValueError, "scores and sel_pages must have rows");
  const uint32_t budget = u32(a[12]), max_pages = u32(a[14]);
  void* s = stream();
  call("aoakv_sparse_decode_layer", [&] {
    return g_lib.sparse_decode_layer(
        ptr(q), ptr(o), ptr(kv), ip, ix, lpl, ptr(meta), mip, mix, log_norm,
        static_cast<float*>(ptr(scores)), (uint32_t)scores.size(-1),
        static_cast<int32_t*>(ptr(sel)), (uint32_t)sel.size(-1), budget, budgets, ptr(ws),
        (size_t)ws.numel(), (uint32_t)q.size(0), max_pages, (uint32_t)q.size(1), d.H, d.D, d.S,
        d.layout, flags, s);
  });
}

// (q, o or None, kv_data, kv_indices, num_kv_pages, kv_last_page_len, layout,
//  causal) -> o
PyObject* prefill_with_paged_kv_cache(PyObject* const* a) {
  const Tensor &q = f16(a[0], "q"), &kv = f16(a[2], "kv_data");
  if (a[1] != Py_None && !THPVariable_Check(a[1]))
    raise(PyExc_TypeError, "o must be a torch.Tensor");
  const int32_t* ix = i32(a[3], "kv_indices");
  const Dims d = cache_dims(kv, a[6]);
  if (q.dim() != 3 || q.size(2) != d.D)
    raise(PyExc_ValueError,
          "q must be [L, Hq, " + std::to_string(d.D) + "], got " + shape_str(q));
  const uint32_t pages = u32(a[4]), last = u32(a[5]), causal = u32(a[7]),
                 N = (uint32_t)q.size(0), Hq = (uint32_t)q.size(1);
  const Tensor o = a[1] == Py_None ? at::empty_like(q) : THPVariable_Unpack(a[1]);
  // split keys: the chunks' partials, from torch's pool on this stream
  size_t n = g_lib.prefill_workspace_size(pages, last, N, causal, Hq, d.D, d.S);
  Tensor ws;
  if (n != 0) {
    try {
      ws = at::empty({(int64_t)n}, q.options().dtype(at::kByte));
    } catch (const c10::OutOfMemoryError&) {
      n = 0;  // no room (136 MB at most): the call runs unsplit
    }
  }
  void* s = stream();
  call("aoakv_prefill_with_paged_kv_cache", [&] {
    return g_lib.prefill_with_workspace(ptr(q), ptr(o), ptr(kv), ix, pages, last, N, causal, Hq,
                                        d.H, d.D, d.S, d.layout, n != 0 ? ptr(ws) : nullptr, n,
                                        s);
  });
  return THPVariable_Wrap(o);
}

// (input, weight, output, epsilon)
void rms_norm_forward(PyObject* const* a) {
  const Tensor &x = f16(a[0], "input"), &w = f16(a[1], "weight"), &o = f16(a[2], "output");
  if (x.dim() == 0) raise(PyExc_ValueError, "input must have a last dimension");
  const int64_t n = x.size(-1);
  if (w.dim() != 1 || w.size(0) != n || o.sizes() != x.sizes())
    raise(PyExc_ValueError, "weight must be [" + std::to_string(n) + "] and output " +
                                shape_str(x) + ", got " + shape_str(w) + " / " + shape_str(o));
  if (n == 0) raise(PyExc_ZeroDivisionError, "integer division or modulo by zero");
  const float eps = f32(a[3]);
  void* s = stream();
  call("aoakv_rms_norm_forward", [&] {
    return g_lib.rms_norm_forward(ptr(x), ptr(w), ptr(o), (uint32_t)(x.numel() / n), (uint32_t)n,
                                  eps, s);
  });
}

// No C++ exception leaves a call: torch's become RuntimeError.
template <auto F, Py_ssize_t N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
  try {
    if (n != N) raise(PyExc_TypeError, "expected " + std::to_string(N) + " arguments");
    if (g_lib.last_error == nullptr) raise(PyExc_RuntimeError, "aoakv._host is not bound");
    if constexpr (std::is_void_v<decltype(F(args))>) {
      F(args);
      Py_RETURN_NONE;
    } else {
      return F(args);
    }
  } catch (const PyErr&) {
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
  } catch (...) {
    PyErr_SetString(PyExc_RuntimeError, "unknown C++ exception");
  }
  return nullptr;
}

// bind(path, AoakvError, ArgumentError): the loaded library's entry points
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  const char* path = n == 3 ? PyUnicode_AsUTF8(args[0]) : nullptr;
  if (path == nullptr) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "bind(path, error, argument error)");
    return nullptr;
  }
  void* h = dlopen(path, RTLD_NOW | RTLD_LOCAL);
  if (h == nullptr) return PyErr_Format(PyExc_ImportError, "%s", dlerror());
  Lib lib;
#define X(f)                                                                                \
  lib.f = reinterpret_cast<decltype(lib.f)>(dlsym(h, "aoakv_" #f));                         \
  if (lib.f == nullptr) return PyErr_Format(PyExc_ImportError, "%s lacks aoakv_" #f, path);
  FOR_EACH_ENTRY(X)
#undef X
  Py_XDECREF(g_error);
  Py_XDECREF(g_arg_error);
  Py_INCREF(g_error = args[1]);
  Py_INCREF(g_arg_error = args[2]);
  g_lib = lib;
  Py_RETURN_NONE;
}

#define ENTRY(f, n) \
  {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(entry<f, n>)), METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(bind)), METH_FASTCALL,
     nullptr},
    ENTRY(append_kv_cache_prefill, 11),
    ENTRY(append_kv_cache_decode, 12),
    ENTRY(rope_append_kv_cache_decode, 15),
    ENTRY(rope_append_kv_cache_prefill, 14),
    ENTRY(estimate_attn_score, 12),
    ENTRY(topk_filtering, 10),
    ENTRY(decode_sparse_attn, 14),
    ENTRY(sparse_decode_layer, 18),
    ENTRY(prefill_with_paged_kv_cache, 8),
    ENTRY(rms_norm_forward, 4),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, g_methods,
                        nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__host() {
  return PyModule_Create(&g_module);
}
