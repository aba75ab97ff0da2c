// The host side of one decode token's operators, for CPython and torch tensors.
//
// A decode step is three to six launches of a few microseconds each, and an operator that checks its tensors, reads
// its controller and calls the library through ctypes costs 6 to 12 us of host time: eager steps over short contexts
// waited for Python.  Each function here does the same checks and the same call in one native function.  It serves
// the ordinary call only: plain tensors on the current device, in the shapes, types and order that the operator
// asks for, a controller of the package's own class, nothing to allocate but the result.  For anything else it
// returns None before it has done anything, and the operator in utils/__init__.py goes its general way, which is
// also the one that says what is wrong.  Nothing is kept between calls: every call reads the controller anew.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cmath>
#include <cstring>

#include "../../include/adamas_hip.h"

namespace {

// ---- names, classes and constants of the package, set once by setup() ----------------------------------------------
PyTypeObject* g_controller_type = nullptr;
PyObject* g_controller_module = nullptr;  // holds CODES_CACHED_BYTES
PyObject* g_all_past = nullptr;           // ALL_PAST_TOKENS

#define ADAMAS_NAMES(X)                                                                                             \
  X(dtype) X(batch_size) X(num_layers) X(num_heads) X(num_kv_heads) X(head_dim) X(page_size) X(max_seq_len)         \
  X(hadamard_scale) X(kv_flags) X(code_flags) X(pool) X(seqs) X(kv) X(codes) X(_table_dev) X(indptr_dev)             \
  X(_seq_lens_dev) X(_host_waits) X(lengths) X(max_pages) X(inference_page_budget)                                   \
  X(topk_dout_buffer) X(topk_dindices_buffer) X(topk_buf) X(_workspace) X(_len_bound) X(_estimate_buf)               \
  X(_estimate_version) X(CODES_CACHED_BYTES)
#define ADAMAS_DECLARE(n) PyObject* s_##n = nullptr;
ADAMAS_NAMES(ADAMAS_DECLARE)
#undef ADAMAS_DECLARE

// A call that is not served is an ordinary one too (the first of a controller, a subclass', one with a numpy integer),
// so every check says no by its result.  An exception costs 3 to 5 us, 60 with cold caches and 0.3 s the first time in
// a process, when the unwinder reads the tables of torch's libraries.
#define ADAMAS_NEED(...)                    \
  do {                                      \
    if (!(__VA_ARGS__)) Py_RETURN_NONE;     \
  } while (0)

struct Ref {  // an owned reference
  PyObject* p = nullptr;
  Ref() = default;
  explicit Ref(PyObject* q) : p(q) {}
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
  ~Ref() { Py_XDECREF(p); }

  bool read(PyObject* o, PyObject* name) {  // an attribute
    Py_XDECREF(p);
    p = PyObject_GetAttr(o, name);
    if (!p) PyErr_Clear();
    return p != nullptr;
  }
};

bool as_long(PyObject* v, long& x) {
  if (!PyLong_CheckExact(v)) return false;
  int over = 0;
  x = PyLong_AsLongAndOverflow(v, &over);
  return over == 0;
}

bool attr_long(PyObject* o, PyObject* name, long& x) {
  Ref v;
  return v.read(o, name) && as_long(v.p, x);
}

// a number that the library takes in 32 bits
template <typename T>
bool attr_u32(PyObject* o, PyObject* name, T& x) {
  long v;
  if (!attr_long(o, name, v) || v < 0 || v > 0x7fffffffL) return false;
  x = static_cast<T>(v);
  return true;
}

// A plain tensor on a GPU (no subclass, no wrapper of a transform, no lazy bits), or null.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  static const c10::DispatchKeySet usual({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA,
                                          c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutocastCUDA});
  const bool ok = t.defined() && t.has_storage() && (t.key_set().raw_repr() & ~usual.raw_repr()) == 0 && t.is_cuda();
  return ok ? &t : nullptr;
}

struct Owned {  // a tensor attribute, kept alive for the call
  Ref ref;
  const at::Tensor* t = nullptr;
  bool read(PyObject* o, PyObject* name) {
    t = ref.read(o, name) ? plain(ref.p) : nullptr;
    return t != nullptr;
  }
  char* data() const { return static_cast<char*>(t->data_ptr()); }
  size_t numel() const { return static_cast<size_t>(t->numel()); }
  const int32_t* words() const { return static_cast<const int32_t*>(t->data_ptr()); }
};

// the current stream, if t lies on the current device
bool stream_of(const at::Tensor& t, adamas_stream_t& s) {
  const auto now = c10::hip::getCurrentHIPStream();
  s = now.stream();
  return now.device_index() == t.get_device();
}

// The controller's numbers and device-side state.
struct Controller {
  PyObject* c;
  long batch, heads, kv_heads, page, max_len, min_len, sum_len;
  bool bounded = false;  // lengths stand in for a bound while a graph is in use
  at::ScalarType dtype;
  Ref pool, seqs;

  bool read(PyObject* obj) {
    c = obj;
    if (Py_TYPE(c) != g_controller_type || c10::impl::TorchDispatchModeTLS::any_modes_set()) return false;
    Ref d, lens, bound;
    long dim;
    if (!d.read(c, s_dtype) || !THPDtype_Check(d.p)) return false;
    dtype = reinterpret_cast<THPDtype*>(d.p)->scalar_type;
    if (!attr_u32(c, s_batch_size, batch) || !attr_u32(c, s_num_heads, heads) ||
        !attr_u32(c, s_num_kv_heads, kv_heads) || !attr_u32(c, s_page_size, page) || !attr_long(c, s_head_dim, dim) ||
        dim != ADAMAS_HEAD_DIM || !pool.read(c, s_pool) || !seqs.read(c, s_seqs) || !lens.read(seqs.p, s_lengths) ||
        !PyList_CheckExact(lens.p) || PyList_GET_SIZE(lens.p) == 0)
      return false;
    sum_len = 0;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(lens.p); ++i) {
      long n;
      if (!as_long(PyList_GET_ITEM(lens.p, i), n)) return false;
      max_len = i ? std::max(max_len, n) : n;
      min_len = i ? std::min(min_len, n) : n;
      sum_len += n;
    }
    if (!bound.read(c, s__len_bound)) return false;
    if (bound.p != Py_None) {
      if (!as_long(bound.p, max_len)) return false;
      bounded = true;
    }
    return max_len >= 0 && max_len <= 0x7fffffffL;
  }

  // the budget of the coming layers
  bool budget(uint32_t& b) const { return attr_u32(c, s_inference_page_budget, b) && b >= 1u; }

  // address of one layer of a pool tensor
  bool layer(const Owned& pool_tensor, PyObject* index, char*& p) const {
    long i;
    const long n = pool_tensor.t->size(0);
    if (!as_long(index, i) || i < -n || i >= n) return false;
    p = pool_tensor.data() + (i < 0 ? i + n : i) * pool_tensor.t->stride(0) * pool_tensor.t->element_size();
    return true;
  }

  // the flag that InferenceController.codes_flags gives
  bool codes_flags(uint32_t budget_now, uint32_t& flag) const {
    long layers, most;
    if (!attr_u32(c, s_num_layers, layers) || !attr_long(g_controller_module, s_CODES_CACHED_BYTES, most))
      return false;
    const long tokens = bounded ? batch * max_len : sum_len;
    const long bytes = layers * (tokens * kv_heads * 2 * ADAMAS_CODE_WORDS +
                                 batch * static_cast<long>(budget_now) * heads * 512);
    flag = bytes <= most ? ADAMAS_F_CODES_CACHED : ADAMAS_F_CODES_STREAMED;
    return true;
  }

  // The current stream, if it is t's device's and lengths and pages need no wait there (PagedSequences.__init__):
  // PagedSequences.launch_addresses sees to the others.
  bool stream(const at::Tensor& t, adamas_stream_t& s) const {
    Ref waits;
    return stream_of(t, s) && waits.read(seqs.p, s__host_waits) &&
           (waits.p == Py_True || (waits.p == Py_False && s == nullptr));
  }

  bool workspace(Owned& ws, uint32_t budget_now) const {  // the controller's, if it is large enough
    long most;
    if (!ws.read(c, s__workspace) || !attr_u32(c, s_max_seq_len, most)) return false;
    const uint32_t b = static_cast<uint32_t>(std::max(1L, std::min(static_cast<long>(budget_now), most)));
    const uint32_t len = static_cast<uint32_t>(std::max(1L, std::min(max_len, most)));
    return ws.numel() >= adamas_workspace_bytes(static_cast<uint32_t>(batch), static_cast<uint32_t>(heads), len, b);
  }
};

bool is_rows(const at::Tensor& t, at::ScalarType dtype, long n, long heads) {
  return t.scalar_type() == dtype && t.dim() == 3 && t.size(0) == n && t.size(1) == heads &&
         t.size(2) == ADAMAS_HEAD_DIM && t.is_contiguous();
}

// the packed code of a query
bool is_code(const at::Tensor& t, const Controller& c) {
  return t.element_size() == 2 && t.dim() == 3 && t.size(0) == c.batch && t.size(1) == c.heads &&
         t.size(2) == ADAMAS_CODE_WORDS && t.is_contiguous();
}

PyObject* failed(const char* what, int code) {
  PyErr_Format(PyExc_RuntimeError, "%s failed with error code %d: %s", what, code, adamas_error_string(code));
  return nullptr;
}

template <typename F>
int released(F&& f) {  // a launch can wait for room in the queue: other threads go on meanwhile
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = f();
  Py_END_ALLOW_THREADS
  return rc;
}

// ---- the operators -------------------------------------------------------------------------------------------------
PyObject* hadamard(PyObject* const* a, Py_ssize_t) {  // x, inplace, scale
  const at::Tensor* x = plain(a[0]);
  const bool inplace = a[1] == Py_True;
  adamas_stream_t s;
  ADAMAS_NEED(x && (inplace || a[1] == Py_False) && PyFloat_CheckExact(a[2]) &&
              !c10::impl::TorchDispatchModeTLS::any_modes_set());
  ADAMAS_NEED((x->scalar_type() == at::kHalf || x->scalar_type() == at::kBFloat16) && x->dim() > 0 &&
              x->size(-1) == ADAMAS_HEAD_DIM && x->is_contiguous() && stream_of(*x, s));
  const at::Tensor out = inplace ? *x : at::empty_like(*x);
  const float scale = static_cast<float>(PyFloat_AS_DOUBLE(a[2]));
  const uint32_t flags = x->scalar_type() == at::kBFloat16 ? ADAMAS_F_BF16 : 0u;
  const void* xp = x->data_ptr();
  void* op = out.data_ptr();
  const uint64_t rows = static_cast<uint64_t>(x->numel()) / ADAMAS_HEAD_DIM;
  const int rc = released([&] { return adamas_hadamard_f(xp, op, rows, scale, flags, s); });
  if (rc) return failed("adamas_hadamard", rc);
  return THPVariable_Wrap(out);  // (in place: the object that was given)
}

PyObject* append_decode(PyObject* const* a, Py_ssize_t) {  // k, v, h, q, controller, layer
  const bool from_h = a[2] != Py_None;
  ADAMAS_NEED(from_h != (a[3] != Py_None));
  const at::Tensor *k = plain(a[0]), *v = plain(a[1]), *x = plain(from_h ? a[2] : a[3]);
  ADAMAS_NEED(k && v && x && !(from_h && x->sizes() == k->sizes()));  // (a prompt's h)
  Controller c;
  ADAMAS_NEED(c.read(a[4]) && c.min_len >= 1);
  const long n = c.batch;
  ADAMAS_NEED(is_rows(*k, c.dtype, n, c.kv_heads) && is_rows(*v, c.dtype, n, c.kv_heads));
  if (!from_h) {
    ADAMAS_NEED(is_rows(*x, c.dtype, n, c.heads));
  } else if (c.heads == c.kv_heads) {
    ADAMAS_NEED(is_rows(*x, c.dtype, 2 * n, c.heads));
  } else {
    ADAMAS_NEED(x->scalar_type() == c.dtype && x->dim() == 2 && x->size(0) == n * (c.heads + c.kv_heads) &&
                x->size(1) == ADAMAS_HEAD_DIM && x->is_contiguous());
  }
  Owned kv, codes, table, indptr, lens;
  Ref scale;
  uint32_t flags;
  char *kv_p, *codes_p;
  adamas_stream_t s;
  ADAMAS_NEED(kv.read(c.pool.p, s_kv) && codes.read(c.pool.p, s_codes) && table.read(c.seqs.p, s__table_dev) &&
              indptr.read(c.seqs.p, s_indptr_dev) && lens.read(c.seqs.p, s__seq_lens_dev));
  ADAMAS_NEED(scale.read(c.c, s_hadamard_scale) && PyFloat_CheckExact(scale.p) && attr_u32(c.c, s_code_flags, flags));
  ADAMAS_NEED(c.layer(kv, a[5], kv_p) && c.layer(codes, a[5], codes_p) && c.stream(*k, s));
  at::Tensor o = at::empty({n, c.heads, ADAMAS_CODE_WORDS}, k->options().dtype(at::kShort));
  const void *kp = k->data_ptr(), *vp = v->data_ptr(), *xp = x->data_ptr();
  void* op = o.data_ptr();
  const int rc = released([&] {
    return adamas_append_decode(from_h ? nullptr : xp, kp, vp, from_h ? xp : nullptr, static_cast<uint16_t*>(op), kv_p,
                                codes_p, table.words(), indptr.words(), lens.words(), static_cast<uint32_t>(n),
                                static_cast<uint32_t>(c.heads), static_cast<uint32_t>(c.kv_heads), ADAMAS_HEAD_DIM,
                                static_cast<uint32_t>(c.page), static_cast<float>(PyFloat_AS_DOUBLE(scale.p)), flags,
                                s);
  });
  if (rc) return failed("adamas_append_decode", rc);
  return THPVariable_Wrap(o);
}

PyObject* estimate(PyObject* const* a, Py_ssize_t) {  // q_code, controller, layer
  const at::Tensor* q = plain(a[0]);
  Controller c;
  ADAMAS_NEED(q && c.read(a[1]));
  ADAMAS_NEED(is_code(*q, c) && c.max_len >= 2);
  Owned codes, table, indptr, lens;
  char* codes_p;
  adamas_stream_t s;
  ADAMAS_NEED(codes.read(c.pool.p, s_codes) && table.read(c.seqs.p, s__table_dev) &&
              indptr.read(c.seqs.p, s_indptr_dev) && lens.read(c.seqs.p, s__seq_lens_dev));
  ADAMAS_NEED(c.layer(codes, a[2], codes_p) && c.stream(*q, s));
  const long n = c.max_len - 1, stride = (n + 7) / 8 * 8;
  at::Tensor buf = at::empty({c.batch, c.heads, stride}, q->options().dtype(at::kHalf));
  const void* qp = q->data_ptr();
  void* bp = buf.data_ptr();
  const int rc = released([&] {
    return adamas_estimate(static_cast<const uint16_t*>(qp), codes_p, table.words(), indptr.words(), lens.words(), bp,
                           c.heads * stride, stride, ADAMAS_DIST_FP16, static_cast<uint32_t>(c.batch),
                           static_cast<uint32_t>(c.heads), static_cast<uint32_t>(c.kv_heads),
                           static_cast<uint32_t>(c.page), static_cast<uint32_t>(c.max_len), s);
  });
  if (rc) return failed("adamas_estimate", rc);
  at::Tensor out = c.batch == 1 ? buf.as_strided({c.heads, n}, {stride, 1})
                                : buf.as_strided({c.batch, c.heads, n}, {c.heads * stride, stride, 1});
  const Ref version(PyLong_FromLongLong(buf._version())), held(THPVariable_Wrap(buf));
  if (!version.p || !held.p || PyObject_SetAttr(c.c, s__estimate_buf, held.p) < 0 ||
      PyObject_SetAttr(c.c, s__estimate_version, version.p) < 0)
    return nullptr;
  return THPVariable_Wrap(out);
}

PyObject* topk(PyObject* const* a, Py_ssize_t) {  // estimate, controller, integer_keys; True when done
  const at::Tensor* est = plain(a[0]);
  Controller c;
  ADAMAS_NEED(est && c.read(a[1]));
  const long rows = c.batch * c.heads;
  ADAMAS_NEED(est->scalar_type() == at::kHalf && (est->dim() == 2 || est->dim() == 3) && est->stride(-1) == 1);
  long row_stride = est->stride(0);
  if (est->dim() == 3) {
    ADAMAS_NEED(est->size(0) == c.batch && est->size(1) == c.heads && est->stride(0) == est->stride(1) * est->size(1));
    row_stride = est->stride(1);
  } else {
    ADAMAS_NEED(est->size(0) == rows);
  }
  uint32_t budget;
  ADAMAS_NEED(c.budget(budget));
  const uint32_t k = budget - 1u;
  const long n = est->size(-1);
  ADAMAS_NEED(n > 0 && (n >= static_cast<long>(k) || c.batch > 1));
  Owned idx, val, scratch, lens;
  long most;
  ADAMAS_NEED(idx.read(c.c, s_topk_dindices_buffer) && val.read(c.c, s_topk_dout_buffer) &&
              scratch.read(c.c, s_topk_buf) && lens.read(c.seqs.p, s__seq_lens_dev) &&
              attr_u32(c.c, s_max_seq_len, most));
  ADAMAS_NEED(scratch.numel() >=
              adamas_topk_workspace_bytes(static_cast<uint32_t>(rows), static_cast<uint32_t>(std::max(n, most)), k));
  bool integer = a[2] == Py_True;
  if (a[2] == Py_None) {
    // views of the buffer that the last estimate filled and that nobody has edited since
    Ref held;
    if (held.read(c.c, s__estimate_buf) && held.p != Py_None) {
      const at::Tensor* buf = plain(held.p);
      long version;
      ADAMAS_NEED(buf && attr_long(c.c, s__estimate_version, version));
      const char* base = static_cast<const char*>(buf->storage().data());
      const char* p = static_cast<const char*>(est->data_ptr());
      integer = static_cast<long>(buf->_version()) == version && base <= p && p < base + buf->storage().nbytes();
    }
  } else {
    ADAMAS_NEED(integer || a[2] == Py_False);
  }
  adamas_stream_t s;
  ADAMAS_NEED(c.stream(*est, s));
  const void* ep = est->data_ptr();
  const int rc = released([&] {
    return adamas_topk(ep, row_stride, static_cast<uint32_t>(n), c.batch > 1 ? lens.words() : nullptr,
                       static_cast<uint32_t>(c.heads), -1, nullptr, 0, static_cast<uint32_t>(rows), k,
                       reinterpret_cast<int32_t*>(idx.data()), val.data(), k,
                       integer ? ADAMAS_KEY_FP16_INT : ADAMAS_KEY_FP16_GENERIC, scratch.data(), scratch.numel(), s);
  });
  if (rc) return failed("adamas_topk", rc);
  Py_RETURN_TRUE;
}

PyObject* sparse_attn(PyObject* const* a, Py_ssize_t) {  // q, controller, layer, indices
  const at::Tensor* q = plain(a[0]);
  Controller c;
  ADAMAS_NEED(q && c.read(a[1]) && is_rows(*q, c.dtype, c.batch, c.heads));
  const int32_t* sel = nullptr;
  long stride = 0, n_sel = 0;
  if (a[3] != Py_None && a[3] != g_all_past) {
    const at::Tensor* t = plain(a[3]);
    ADAMAS_NEED(t && t->scalar_type() == at::kInt && t->dim() == 2 && t->is_contiguous() &&
                t->size(0) == c.batch * c.heads);
    sel = static_cast<const int32_t*>(t->data_ptr());
    stride = t->stride(0);
    n_sel = t->size(1);
  }
  Ref b;
  uint32_t budget = 1, flags;
  Owned kv, table, indptr, lens, ws;
  char* kv_p;
  adamas_stream_t s;
  ADAMAS_NEED(b.read(c.c, s_inference_page_budget) && (b.p == Py_None || c.budget(budget)) && c.workspace(ws, budget));
  ADAMAS_NEED(kv.read(c.pool.p, s_kv) && table.read(c.seqs.p, s__table_dev) && indptr.read(c.seqs.p, s_indptr_dev) &&
              lens.read(c.seqs.p, s__seq_lens_dev));
  ADAMAS_NEED(attr_u32(c.c, s_kv_flags, flags) && c.layer(kv, a[2], kv_p) && c.stream(*q, s));
  at::Tensor o = at::empty_like(*q);
  const void* qp = q->data_ptr();
  void* op = o.data_ptr();
  const int rc = released([&] {
    return adamas_sparse_decode_f(qp, kv_p, table.words(), indptr.words(), lens.words(), sel, stride,
                                  static_cast<uint32_t>(n_sel), op, ws.data(), ws.numel(),
                                  static_cast<uint32_t>(c.batch), static_cast<uint32_t>(c.heads),
                                  static_cast<uint32_t>(c.kv_heads), ADAMAS_HEAD_DIM, static_cast<uint32_t>(c.page),
                                  static_cast<float>(1.0 / std::sqrt(128.0)), static_cast<uint32_t>(c.max_len), flags,
                                  s);
  });
  if (rc) return failed("adamas_sparse_decode", rc);
  return THPVariable_Wrap(o);
}

PyObject* step(PyObject* const* a, Py_ssize_t) {  // q, q_code, controller, layer (no positions asked for)
  const at::Tensor *q = plain(a[0]), *code = plain(a[1]);
  Controller c;
  ADAMAS_NEED(q && code && c.read(a[2]));
  ADAMAS_NEED(is_rows(*q, c.dtype, c.batch, c.heads) && is_code(*code, c));
  uint32_t budget, flags, cached, pages;
  Owned kv, codes, table, indptr, lens, ws;
  char *kv_p, *codes_p;
  adamas_stream_t s;
  ADAMAS_NEED(c.budget(budget) && c.workspace(ws, budget));
  ADAMAS_NEED(kv.read(c.pool.p, s_kv) && codes.read(c.pool.p, s_codes) && table.read(c.seqs.p, s__table_dev) &&
              indptr.read(c.seqs.p, s_indptr_dev) && lens.read(c.seqs.p, s__seq_lens_dev));
  ADAMAS_NEED(attr_u32(c.c, s_kv_flags, flags) && c.codes_flags(budget, cached) &&
              attr_u32(c.seqs.p, s_max_pages, pages));
  ADAMAS_NEED(c.layer(kv, a[3], kv_p) && c.layer(codes, a[3], codes_p) && c.stream(*q, s));
  at::Tensor o = at::empty_like(*q);
  const void *qp = q->data_ptr(), *cp = code->data_ptr();
  void* op = o.data_ptr();
  const int rc = released([&] {
    return adamas_decode_step_f(qp, cp, kv_p, codes_p, table.words(), indptr.words(), lens.words(), budget, op, nullptr,
                                ws.data(), ws.numel(), static_cast<uint32_t>(c.batch), static_cast<uint32_t>(c.heads),
                                static_cast<uint32_t>(c.kv_heads), ADAMAS_HEAD_DIM, static_cast<uint32_t>(c.page),
                                static_cast<float>(1.0 / std::sqrt(128.0)), static_cast<uint32_t>(c.max_len), pages,
                                flags | cached, s);
  });
  if (rc) return failed("adamas_decode_step", rc);
  return THPVariable_Wrap(o);
}

template <PyObject* (*F)(PyObject* const*, Py_ssize_t), int kArgs>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != kArgs) {
    PyErr_Format(PyExc_TypeError, "%d arguments expected, got %zd", kArgs, n);
    return nullptr;
  }
  return F(args, n);
  END_HANDLE_TH_ERRORS
}

PyObject* setup(PyObject*, PyObject* const* args, Py_ssize_t n) {  // InferenceController, its module, ALL_PAST_TOKENS
  if (n != 3 || !PyType_Check(args[0])) {
    PyErr_SetString(PyExc_TypeError, "setup(controller class, its module, marker) expected");
    return nullptr;
  }
  for (Py_ssize_t i = 0; i < n; ++i) Py_INCREF(args[i]);
  g_controller_type = reinterpret_cast<PyTypeObject*>(args[0]);
  g_controller_module = args[1];
  g_all_past = args[2];
  Py_RETURN_NONE;
}

#define ADAMAS_ENTRY(name, f, n) \
  {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<f, n>)), METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {
    ADAMAS_ENTRY("hadamard", hadamard, 3),
    ADAMAS_ENTRY("append_decode", append_decode, 6),
    ADAMAS_ENTRY("estimate", estimate, 3),
    ADAMAS_ENTRY("topk", topk, 3),
    ADAMAS_ENTRY("sparse_attn", sparse_attn, 4),
    ADAMAS_ENTRY("step", step, 4),
    {"setup", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&setup)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "adamas_host", nullptr, -1, g_methods,
                        nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_adamas_host(void) {
  // private headers: only the torch that this was built with
  const Ref torch(PyImport_ImportModule("torch"));
  if (!torch.p) return nullptr;
  const Ref version(PyObject_GetAttrString(torch.p, "__version__"));
  if (!version.p) return nullptr;
  const Ref text(PyObject_Str(version.p));
  const char* now = text.p ? PyUnicode_AsUTF8(text.p) : nullptr;
  if (!now) return nullptr;
  if (std::strcmp(now, ADAMAS_TORCH_VERSION) != 0) {
    PyErr_Format(PyExc_ImportError, "it was built for torch %s, this is %s", ADAMAS_TORCH_VERSION, now);
    return nullptr;
  }
#define ADAMAS_INTERN(n) \
  if (!(s_##n = PyUnicode_InternFromString(#n))) return nullptr;
  ADAMAS_NAMES(ADAMAS_INTERN)
#undef ADAMAS_INTERN
  return PyModule_Create(&g_module);
}
