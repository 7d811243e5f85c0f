// The wrappers' common case in native code: one call takes the torch tensors,
// checks them, allocates outputs and workspace and makes the C-ABI call of
// libkvdec.so (include/kvdec.h) on torch's current stream.
//
// A decode step at the benchmark's small windows runs 4 to 6 us on the GPU;
// the same checks, allocations and ctypes conversions in Python take 10 to 35
// us, so the GPU waits for the host (KIVI decode, B=32, W=256: 23 us a call
// for a 6 us kernel).  The functions here accept exactly the calls described
// at each one and return None for everything else (other argument types,
// tensor subclasses, functorch or fake tensors, an active torch mode, and
// every argument that the wrapper refuses); the wrapper then goes through its
// own checks, which are also where the error messages come from.

#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TracerMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/generated/variable_factories.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <algorithm>
#include <climits>
#include <initializer_list>

#include "kvdec.h"

namespace {

using at::Tensor;
using Shape = std::initializer_list<int64_t>;

#define KVDEC_HOST_FUNCTIONS(X)                                                                  \
  X(kvdec_workspace_bytes) X(kvdec_dense_decode) X(kvdec_sparse_decode) X(kvdec_paged_decode)    \
  X(kvdec_sparse_decode_varlen) X(kvdec_quantize_k) X(kvdec_quantize_v) X(kvdec_sparse_decode_kivi) \
  X(kvdec_sparse_decode_kivi_varlen) X(kvdec_sparse_decode_kivi_typed) X(kvdec_build_kivi_cache) \
  X(kvdec_kivi_stream_step_decode)

// The library's entry points, resolved once by bind().
struct Lib {
#define KVDEC_MEMBER(name) decltype(&::name) name = nullptr;
  KVDEC_HOST_FUNCTIONS(KVDEC_MEMBER)
#undef KVDEC_MEMBER
};
Lib lib;
PyObject* check_rc = nullptr;   // _kvdec.check: raises for a nonzero return code

// -- arguments ----------------------------------------------------------------

bool to_i64(PyObject* o, int64_t& v) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}
bool to_i32(PyObject* o, int32_t& v) {
  int64_t x;
  if (!to_i64(o, x) || x < INT32_MIN || x > INT32_MAX) return false;
  v = (int32_t)x;
  return true;
}
bool to_f32(PyObject* o, float& v) {
  if (!PyFloat_CheckExact(o)) return false;
  v = (float)PyFloat_AS_DOUBLE(o);
  return true;
}
bool fits_i32(int64_t x) { return x >= 0 && x <= INT32_MAX; }

// No tracing and no Python-level mode that would have to see the allocations.
bool plain_mode() {
  return !at::impl::torch_function_mode_enabled() &&
         !c10::impl::TorchDispatchModeTLS::any_modes_set(/*skip_infra_modes=*/false) &&
         !at::tracer::impl::is_dispatch_enabled();
}

const c10::DispatchKeySet kWrapperKeys({
    c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::PythonDispatcher,
    c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Batched,
    c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
    c10::DispatchKey::ZeroTensor});

// A plain strided GPU tensor (torch.Tensor or Parameter itself), or null.
const Tensor* gpu_tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != c10::kStrided || t.key_set().has_any(kWrapperKeys))
    return nullptr;
  return &t;
}
bool shaped(const Tensor& t, Shape s) { return t.sizes() == at::IntArrayRef(s); }

// kvdec element type of an attention tensor, -1 for others
int elt(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kHalf: return KVDEC_F16;
    case at::kFloat: return KVDEC_F32;
    case at::kBFloat16: return KVDEC_BF16;
    default: return -1;
  }
}

// q: [B, H, D], contiguous, of an attention element type
const Tensor* query(PyObject* o) {
  const Tensor* q = gpu_tensor(o);
  return q && q->dim() == 3 && elt(*q) >= 0 && q->is_contiguous() && fits_i32(q->size(1)) && fits_i32(q->size(2))
             ? q : nullptr;
}

// Contiguous tensor of a type and shape on a device.
const Tensor* exactly(PyObject* o, at::ScalarType type, Shape s, c10::Device dev) {
  const Tensor* t = gpu_tensor(o);
  return t && t->scalar_type() == type && shaped(*t, s) && t->device() == dev && t->is_contiguous() ? t : nullptr;
}

// seq_len: an int, or a [B] int32 tensor of per-sequence lengths.
struct SeqLen {
  int64_t n = 0;
  const Tensor* t = nullptr;
  bool parse(PyObject* o, int64_t B, c10::Device dev) {
    if (to_i64(o, n)) return true;
    t = exactly(o, at::kInt, {B}, dev);
    return t != nullptr;
  }
  const int32_t* lens() const { return t ? (const int32_t*)t->data_ptr() : nullptr; }
};

void* stream(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor empty(at::IntArrayRef s, const Tensor& like, at::ScalarType type) {
  return torch::empty(s, at::TensorOptions().dtype(type).device(like.device()));
}
Tensor workspace(size_t bytes, const Tensor& like) {
  return bytes ? empty({(int64_t)bytes}, like, at::kByte) : Tensor();
}
void* ptr(const Tensor& t) { return t.defined() && t.numel() ? t.data_ptr() : nullptr; }

PyObject* none() { Py_RETURN_NONE; }

// The result of a call: the output, or the exception check_rc raises.
PyObject* done(int rc, const char* what, Tensor& o) {
  if (rc == 0) return THPVariable_Wrap(std::move(o));
  PyObject* r = PyObject_CallFunction(check_rc, "is", rc, what);
  Py_XDECREF(r);
  return r ? none() : nullptr;
}

// The GIL is released from here to the end of the scope (a launch can wait
// for room in its queue, an allocation for the device).
struct NoGil {
  PyThreadState* s = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(s); }
};

// -- decode -------------------------------------------------------------------

// sparse(q, k, v, seq_len, window, sink, layout, sm_scale): contiguous
// [B, KVH, sink + window, D] caches of q's type.
PyObject* sparse(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int32_t window, sink, layout;
  float scale;
  const Tensor* q;
  if (n != 8 || !plain_mode() || !(q = query(a[0])) || !to_i32(a[4], window) || !to_i32(a[5], sink) ||
      !to_i32(a[6], layout) || !to_f32(a[7], scale) || window < 0 || sink < 0)
    return none();
  const int64_t B = q->size(0), H = q->size(1), D = q->size(2), slots = (int64_t)window + sink;
  const Tensor* k0 = gpu_tensor(a[1]);
  if (!k0 || k0->dim() != 4 || !fits_i32(k0->size(1))) return none();
  const int64_t KVH = k0->size(1);
  const Tensor* k = exactly(a[1], q->scalar_type(), {B, KVH, slots, D}, q->device());
  const Tensor* v = exactly(a[2], q->scalar_type(), {B, KVH, slots, D}, q->device());
  SeqLen len;
  if (!k || !v || !len.parse(a[3], B, q->device())) return none();
  Tensor o;
  int rc;
  {
    NoGil no_gil;
    o = torch::empty_like(*q);
    const size_t bytes = lib.kvdec_workspace_bytes(KVDEC_KIND_SPARSE, B, (int)H, (int)KVH, slots, (int)D);
    const Tensor ws = workspace(bytes, *q);
    rc = len.t ? lib.kvdec_sparse_decode_varlen(q->data_ptr(), k->data_ptr(), v->data_ptr(), o.data_ptr(),
                                                len.lens(), elt(*q), B, (int)H, (int)KVH, window, sink, layout,
                                                scale, ptr(ws), bytes, stream(*q))
               : lib.kvdec_sparse_decode(q->data_ptr(), k->data_ptr(), v->data_ptr(), o.data_ptr(), elt(*q), B,
                                         (int)H, (int)KVH, len.n, window, sink, layout, scale, ptr(ws), bytes,
                                         stream(*q));
  }
  return done(rc, "sparse_decode_attention", o);
  END_HANDLE_TH_ERRORS
}

// dense(q, k, v, seq_len, sm_scale): [B, KVH, L, D] caches of q's type, either
// contiguous with one length, or (fp16) of common strides or with lengths.
PyObject* dense(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  float scale;
  const Tensor *q, *k, *v;
  SeqLen len;
  if (n != 5 || !plain_mode() || !(q = query(a[0])) || !(k = gpu_tensor(a[1])) || !(v = gpu_tensor(a[2])) ||
      k->dim() != 4 || !to_f32(a[4], scale) || !len.parse(a[3], q->size(0), q->device()))
    return none();
  const int64_t B = q->size(0), H = q->size(1), D = q->size(2), KVH = k->size(1), L = k->size(2);
  const bool one = !len.t && k->is_contiguous() && v->is_contiguous();
  if (!shaped(*k, {B, KVH, L, D}) || !shaped(*v, {B, KVH, L, D}) || k->scalar_type() != q->scalar_type() ||
      v->scalar_type() != q->scalar_type() || k->device() != q->device() || v->device() != q->device() ||
      !fits_i32(KVH) || (!len.t && len.n != L) ||
      (!one && (elt(*q) != KVDEC_F16 || k->strides() != v->strides() || k->stride(3) != 1)))
    return none();
  Tensor o;
  int rc;
  {
    NoGil no_gil;
    o = torch::empty_like(*q);
    const size_t bytes = lib.kvdec_workspace_bytes(KVDEC_KIND_DENSE, B, (int)H, (int)KVH, L, (int)D);
    const Tensor ws = workspace(bytes, *q);
    rc = one ? lib.kvdec_dense_decode(q->data_ptr(), k->data_ptr(), v->data_ptr(), o.data_ptr(), elt(*q), B,
                                      (int)H, (int)KVH, L, (int)D, scale, ptr(ws), bytes, stream(*q))
             : lib.kvdec_paged_decode(q->data_ptr(), k->data_ptr(), v->data_ptr(), nullptr, len.lens(),
                                      o.data_ptr(), KVDEC_F16, B, (int)H, (int)KVH, (int)D, L, 0, 0, 0,
                                      k->stride(0), k->stride(2), k->stride(1), scale, ptr(ws), bytes, stream(*q));
  }
  return done(rc, "dense_decode_attention", o);
  END_HANDLE_TH_ERRORS
}

// paged(q, k_pages, v_pages, block_table, seq_lens, max_seq_len, sm_scale,
// head_major): fp16 pages of common strides, an int for the longest length.
PyObject* paged(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  float scale;
  int64_t longest;
  const Tensor *q, *k, *v, *table, *lens;
  if (n != 8 || !plain_mode() || !(q = query(a[0])) || elt(*q) != KVDEC_F16 || !(k = gpu_tensor(a[1])) ||
      !(v = gpu_tensor(a[2])) || !(table = gpu_tensor(a[3])) || !to_i64(a[5], longest) || !to_f32(a[6], scale) ||
      k->dim() != 4 || table->dim() != 2)
    return none();
  const bool hnd = a[7] == Py_True;
  const int64_t B = q->size(0), H = q->size(1), D = q->size(2);
  const int rows = hnd ? 2 : 1, heads = hnd ? 1 : 2;
  if (!(lens = exactly(a[4], at::kInt, {B}, q->device())) || k->scalar_type() != at::kHalf ||
      v->scalar_type() != at::kHalf || k->device() != q->device() || v->device() != q->device() ||
      k->size(3) != D || k->sizes() != v->sizes() || k->strides() != v->strides() || k->stride(3) != 1 ||
      table->scalar_type() != at::kInt || table->device() != q->device() || !table->is_contiguous() ||
      table->size(0) != B || !fits_i32(k->size(heads)) || !fits_i32(k->size(rows)) || !fits_i32(table->size(1)))
    return none();
  longest = std::max<int64_t>(longest, 1);
  const int KVH = (int)k->size(heads);
  Tensor o;
  int rc;
  {
    NoGil no_gil;
    o = torch::empty_like(*q);
    const size_t bytes = lib.kvdec_workspace_bytes(KVDEC_KIND_DENSE, B, (int)H, KVH, longest, (int)D);
    const Tensor ws = workspace(bytes, *q);
    rc = lib.kvdec_paged_decode(q->data_ptr(), k->data_ptr(), v->data_ptr(), (const int32_t*)table->data_ptr(),
                                (const int32_t*)lens->data_ptr(), o.data_ptr(), KVDEC_F16, B, (int)H, KVH, (int)D,
                                longest, (int)k->size(rows), (int)table->size(1), k->size(0), k->stride(0),
                                k->stride(rows), k->stride(heads), scale, ptr(ws), bytes, stream(*q));
  }
  return done(rc, "paged_decode_attention", o);
  END_HANDLE_TH_ERRORS
}

// kivi(q, k_res, v_res, 12 quantized tensors, seq_len, window, sink, residual,
// group, bits, sm_scale)
PyObject* kivi(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int32_t window, sink, R, G, bits;
  float scale;
  const Tensor *q, *kr;
  SeqLen len;
  if (n != 22 || !plain_mode() || !(q = query(a[0])) || !(kr = gpu_tensor(a[1])) || kr->dim() != 4 ||
      !len.parse(a[15], q->size(0), q->device()) || !to_i32(a[16], window) || !to_i32(a[17], sink) ||
      !to_i32(a[18], R) || !to_i32(a[19], G) || !to_i32(a[20], bits) || !to_f32(a[21], scale))
    return none();
  const int64_t B = q->size(0), H = q->size(1), D = q->size(2), KVH = kr->size(1);
  if (window < 1 || R < 0 || bits < 1 || bits > 8 || G < 1 || D % G || G % (8 / bits) || !fits_i32(KVH) ||
      elt(*kr) < 0)
    return none();
  const int64_t pf = 8 / bits, res = std::min(window, R), old = window - res;
  const c10::Device dev = q->device();
  const Tensor* vr;
  if (!(kr = exactly(a[1], kr->scalar_type(), {B, KVH, res, D}, dev)) ||
      !(vr = exactly(a[2], kr->scalar_type(), {B, KVH, res, D}, dev)))
    return none();
  const int64_t shapes[12][2] = {
      {G / pf, D}, {1, D}, {1, D}, {G, D / pf}, {G, D / G}, {G, D / G},
      {old / pf, D}, {old / G, D}, {old / G, D}, {old, D / pf}, {old, D / G}, {old, D / G}};
  const void* parts[12];
  for (int i = 0; i < 12; ++i) {
    const Tensor* t = exactly(a[3 + i], i % 3 == 0 ? at::kByte : at::kHalf,
                              {B, KVH, shapes[i][0], shapes[i][1]}, dev);
    if (!t) return none();
    parts[i] = ptr(*t);
  }
  Tensor o;
  int rc;
  {
    NoGil no_gil;
    o = torch::empty_like(*q);
    if (elt(*q) != KVDEC_F16 || elt(*kr) != KVDEC_F16) {
      rc = lib.kvdec_sparse_decode_kivi_typed(q->data_ptr(), kr->data_ptr(), vr->data_ptr(), parts, o.data_ptr(),
                                              elt(*q), elt(*kr), len.lens(), B, (int)H, (int)KVH,
                                              len.t ? 1 : len.n, window, sink, R, G, bits, scale, stream(*q));
    } else if (len.t) {
      rc = lib.kvdec_sparse_decode_kivi_varlen(q->data_ptr(), kr->data_ptr(), vr->data_ptr(), parts, o.data_ptr(),
                                               len.lens(), B, (int)H, (int)KVH, window, sink, R, G, bits, scale,
                                               stream(*q));
    } else {
      const size_t bytes = lib.kvdec_workspace_bytes(KVDEC_KIND_KIVI_SPLIT, B, (int)H, (int)KVH, old, (int)D);
      const Tensor ws = workspace(bytes, *q);
      rc = lib.kvdec_sparse_decode_kivi(q->data_ptr(), kr->data_ptr(), vr->data_ptr(), parts, o.data_ptr(), B,
                                        (int)H, (int)KVH, len.n, window, sink, R, G, bits, scale, ptr(ws), bytes,
                                        stream(*q));
    }
  }
  return done(rc, "sparse_decode_attention_quantized", o);
  END_HANDLE_TH_ERRORS
}

// step_attend(tensors, q, k_new, v_new, active, appended, arrive, plan, ring,
// sink, residual, n_groups, cap, group, bits, sm_scale): KiviStreamBatch's
// step with contiguous fp16 tokens and an int32 (or no) mask.
PyObject* step_attend(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  static const char* kNames[14] = {
      "k_ring", "v_ring", "k_sink_packed", "k_sink_scale", "k_sink_zero", "v_sink_packed", "v_sink_scale",
      "v_sink_zero", "k_win_packed", "k_win_scale", "k_win_zero", "v_win_packed", "v_win_scale", "v_win_zero"};
  static PyObject* keys[14];
  if (!keys[13])
    for (int i = 0; i < 14; ++i)
      if (!keys[i] && !(keys[i] = PyUnicode_InternFromString(kNames[i]))) return nullptr;
  int32_t geo[6];   // sink, residual, n_groups, cap, group, bits
  float scale;
  const Tensor* q;
  if (n != 16 || !plain_mode() || !PyDict_CheckExact(a[0]) || !(q = query(a[1])) || elt(*q) != KVDEC_F16 ||
      !to_f32(a[15], scale))
    return none();
  for (int i = 0; i < 6; ++i)
    if (!to_i32(a[9 + i], geo[i])) return none();
  // the cache's tensors, held until the launch: the dict lends them, and a
  // thread may replace an entry while the GIL is released
  Tensor t[14];
  for (int i = 0; i < 14; ++i) {
    PyObject* x = PyDict_GetItem(a[0], keys[i]);
    const Tensor* g = x ? gpu_tensor(x) : nullptr;
    if (!g) return none();
    t[i] = *g;
  }
  if (t[0].dim() != 4) return none();
  const c10::Device dev = t[0].device();
  const int64_t B = t[0].size(0), KVH = t[0].size(1), D = t[0].size(3), H = q->size(1);
  const Tensor* tok[2];
  for (int i = 0; i < 2; ++i)
    if (!(tok[i] = gpu_tensor(a[2 + i])) || tok[i]->scalar_type() != at::kHalf || !tok[i]->is_contiguous() ||
        tok[i]->numel() != B * KVH * D || tok[i]->device() != dev)
      return none();
  const Tensor *act = nullptr, *st[4];
  if (a[4] != Py_None && !(act = exactly(a[4], at::kInt, {B}, dev))) return none();
  for (int i = 0; i < 4; ++i)
    if (!(st[i] = gpu_tensor(a[5 + i])) || st[i]->device() != dev) return none();
  if (!shaped(*q, {B, H, D}) || q->device() != dev || !fits_i32(KVH)) return none();
  const void* parts[12];
  for (int i = 0; i < 12; ++i) parts[i] = ptr(t[2 + i]);
  int32_t* state[4];
  for (int i = 0; i < 4; ++i) state[i] = (int32_t*)st[i]->data_ptr();
  void* rings[2] = {t[0].data_ptr(), t[1].data_ptr()};
  Tensor o;
  int rc;
  {
    NoGil no_gil;
    o = torch::empty_like(*q);
    rc = lib.kvdec_kivi_stream_step_decode(
        q->data_ptr(), tok[0]->data_ptr(), tok[1]->data_ptr(), rings[0], rings[1], (void* const*)parts, o.data_ptr(),
        state[0], act ? (const int32_t*)act->data_ptr() : nullptr, state[1], state[2], state[3], B, (int)H,
        (int)KVH, geo[0], geo[1], geo[2], geo[3], geo[4], geo[5], scale, stream(*q));
  }
  return done(rc, "KiviStreamBatch.step_attend", o);
  END_HANDLE_TH_ERRORS
}

// -- quantizers -----------------------------------------------------------------

// quantize(x, group, bits, values): a contiguous non-empty [B, KVH, n, D];
// K per channel over `group` tokens, V (values) per token over `group` channels.
PyObject* quantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int32_t G, bits;
  const Tensor* x;
  if (n != 4 || !plain_mode() || !(x = gpu_tensor(a[0])) || !to_i32(a[1], G) || !to_i32(a[2], bits) ||
      x->dim() != 4 || elt(*x) < 0 || !x->is_contiguous() || G < 1 || bits < 1 || bits > 8)
    return none();
  const bool values = a[3] == Py_True;
  const int64_t B = x->size(0), KVH = x->size(1), len = x->size(2), D = x->size(3), pf = 8 / bits;
  if (len == 0 || (values ? D : len) % G || !fits_i32(KVH) || !fits_i32(D)) return none();
  Tensor out[3];
  int rc;
  {
    NoGil no_gil;
    const int64_t rows = values ? len : len / G, cols = values ? D / G : D;
    out[0] = empty({B, KVH, values ? len : len / pf, values ? D / pf : D}, *x, at::kByte);
    out[1] = empty({B, KVH, rows, cols}, *x, at::kHalf);
    out[2] = empty({B, KVH, rows, cols}, *x, at::kHalf);
    rc = (values ? lib.kvdec_quantize_v : lib.kvdec_quantize_k)(
        x->data_ptr(), elt(*x), out[0].data_ptr(), out[1].data_ptr(), out[2].data_ptr(), B, (int)KVH, len, (int)D,
        G, bits, stream(*x));
  }
  if (rc) return done(rc, values ? "quantize_v_cache" : "quantize_k_cache", out[0]);
  PyObject* r = PyTuple_New(3);
  for (int i = 0; r && i < 3; ++i) {
    PyObject* t = THPVariable_Wrap(std::move(out[i]));
    if (!t) {
      Py_DECREF(r);
      return nullptr;
    }
    PyTuple_SET_ITEM(r, i, t);
  }
  return r;
  END_HANDLE_TH_ERRORS
}

// build(k, v, residual_size, sink, group, bits, residual_fp16): contiguous
// [B, KVH, n, D] caches of one type; residual of the same type or fp16.
PyObject* build(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  static const char* kNames[14] = {
      "k_residual", "v_residual", "k_sink_packed", "k_sink_scale", "k_sink_zero", "v_sink_packed", "v_sink_scale",
      "v_sink_zero", "k_win_packed", "k_win_scale", "k_win_zero", "v_win_packed", "v_win_scale", "v_win_zero"};
  int32_t R, sink, G, bits;
  const Tensor *k, *v;
  if (n_args != 7 || !plain_mode() || !(k = gpu_tensor(a[0])) || !(v = gpu_tensor(a[1])) || !to_i32(a[2], R) ||
      !to_i32(a[3], sink) || !to_i32(a[4], G) || !to_i32(a[5], bits) || k->dim() != 4 || elt(*k) < 0 ||
      v->scalar_type() != k->scalar_type() || v->sizes() != k->sizes() || v->device() != k->device() ||
      !k->is_contiguous() || !v->is_contiguous())
    return none();
  const int64_t B = k->size(0), KVH = k->size(1), n = k->size(2), D = k->size(3), P = 8 / bits;
  if (sink < 1 || sink > G || n <= sink || R < 1 || !fits_i32(KVH) || !fits_i32(n) || !fits_i32(D)) return none();
  const int64_t res = std::min<int64_t>(R, n - sink), old = n - sink - res;
  if (old % G) return none();
  const at::ScalarType rt = a[6] == Py_True ? at::kHalf : k->scalar_type();
  const int64_t shapes[14][2] = {
      {res, D}, {res, D}, {G / P, D}, {1, D}, {1, D}, {G, D / P}, {G, D / G}, {G, D / G},
      {old / P, D}, {old / G, D}, {old / G, D}, {old, D / P}, {old, D / G}, {old, D / G}};
  Tensor out[14];
  int rc;
  {
    NoGil no_gil;
    void* parts[14];
    for (int i = 0; i < 14; ++i) {
      const at::ScalarType type = i < 2 ? rt : (i - 2) % 3 == 0 ? at::kByte : at::kHalf;
      out[i] = empty({B, KVH, shapes[i][0], shapes[i][1]}, *k, type);
      parts[i] = ptr(out[i]);
    }
    rc = lib.kvdec_build_kivi_cache(k->data_ptr(), v->data_ptr(), elt(*k), elt(out[0]), B, (int)KVH, (int)n, (int)D,
                                    sink, R, G, bits, parts, stream(*k));
  }
  if (rc) return done(rc, "build_quantized_kv_cache", out[0]);
  PyObject* d = PyDict_New();
  for (int i = 0; d && i < 14; ++i) {
    PyObject* t = THPVariable_Wrap(std::move(out[i]));
    if (!t || PyDict_SetItemString(d, kNames[i], t)) Py_CLEAR(d);
    Py_XDECREF(t);
  }
  return d;
  END_HANDLE_TH_ERRORS
}

// -- module ---------------------------------------------------------------------

// bind(path, check): the loaded libkvdec.so and _kvdec.check.
PyObject* bind(PyObject*, PyObject* args) {
  const char* path;
  PyObject* check;
  if (!PyArg_ParseTuple(args, "sO", &path, &check)) return nullptr;
  void* so = dlopen(path, RTLD_NOW | RTLD_LOCAL);
  if (!so) return PyErr_Format(PyExc_ImportError, "%s", dlerror());
#define KVDEC_RESOLVE(name)                                   \
  lib.name = reinterpret_cast<decltype(lib.name)>(dlsym(so, #name)); \
  if (!lib.name) return PyErr_Format(PyExc_ImportError, "%s has no " #name, path);
  KVDEC_HOST_FUNCTIONS(KVDEC_RESOLVE)
#undef KVDEC_RESOLVE
  Py_INCREF(check);
  Py_XDECREF(check_rc);
  check_rc = check;
  return none();
}

#define KVDEC_FAST(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    KVDEC_FAST(sparse), KVDEC_FAST(dense), KVDEC_FAST(paged), KVDEC_FAST(kivi), KVDEC_FAST(step_attend),
    KVDEC_FAST(quantize), KVDEC_FAST(build), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_kvdec_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__kvdec_host() {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION)) Py_CLEAR(m);
  return m;
}
