// Direct calls of the C ABI from Python on torch tensors (module
// litevllm._native): per-call checks, output allocation, scratch lookup and
// the library call in one step.
//
// Every function takes the arguments of the wrapper of the same name in
// litevllm/ops.py, in order, and returns the wrapper's result -- or None if
// any argument is not of the plain accepted form (a tensor on another
// device, a shape, stride or dtype the wrapper would reject, a subclass),
// having launched nothing; the wrapper then goes through its own checks,
// which name the fault.  The conditions here are those checks, so a call that
// reaches the library satisfies them all.  A decode step of a small batch
// spends most of its time in the host call, not on the GPU: one
// paged-attention call through the Python checks and ctypes takes 14.5 us,
// the kernels of a short context 8.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>

#include "litevllm_hip.h"

namespace {

// Entry points of liblitevllm_hip.so, bound once by bind().
struct Api {
  decltype(&lv_last_error) last_error;
  decltype(&lv_kv_scatter) kv_scatter;
  decltype(&lv_paged_attention_workspace_size) attention_ws;
  decltype(&lv_paged_attention_split_workspace_size) split_ws;
  decltype(&lv_paged_attention) attention;
  decltype(&lv_paged_attention_prefix_workspace_size) prefix_ws;
  decltype(&lv_paged_attention_prefix) attention_prefix;
  decltype(&lv_sample_workspace_size) sample_ws;
  decltype(&lv_sample) sample;
  decltype(&lv_add_rms_norm) add_rms_norm;
  decltype(&lv_qk_norm_rope_cache) qk_norm_rope_cache;
  decltype(&lv_silu_mul) silu_mul;
  decltype(&lv_linear_one_round) linear_one_round;
  decltype(&lv_linear) linear;
  decltype(&lv_linear_f32) linear_f32;
};
Api api{};

constexpr const char* kNames[] = {
    "lv_last_error", "lv_kv_scatter", "lv_paged_attention_workspace_size",
    "lv_paged_attention_split_workspace_size", "lv_paged_attention",
    "lv_paged_attention_prefix_workspace_size", "lv_paged_attention_prefix",
    "lv_sample_workspace_size", "lv_sample", "lv_add_rms_norm", "lv_qk_norm_rope_cache",
    "lv_silu_mul", "lv_linear_one_round", "lv_linear", "lv_linear_f32"};
constexpr size_t kNumNames = sizeof(kNames) / sizeof(kNames[0]);
static_assert(sizeof(Api) == kNumNames * sizeof(void*), "one pointer per name");

PyObject* workspaces;    // ops._workspaces: {(device index, stream, kind): uint8 tensor}
PyObject *kind_attn, *kind_prefix;

// bind({name: address}, workspaces): the addresses ctypes resolved, and the
// wrappers' scratch buffers.
PyObject* bind(PyObject*, PyObject* args) {
  PyObject *dict, *pool;
  if (!PyArg_ParseTuple(args, "O!O!", &PyDict_Type, &dict, &PyDict_Type, &pool)) return nullptr;
  void* p[kNumNames];
  for (size_t i = 0; i < kNumNames; ++i) {
    PyObject* v = PyDict_GetItemString(dict, kNames[i]);
    p[i] = v ? PyLong_AsVoidPtr(v) : nullptr;
    if (!p[i]) {
      if (!PyErr_Occurred())
        PyErr_Format(PyExc_RuntimeError, "no address for %s", kNames[i]);
      return nullptr;
    }
  }
  if (!kind_attn) kind_attn = PyUnicode_InternFromString("attn");
  if (!kind_prefix) kind_prefix = PyUnicode_InternFromString("prefix");
  if (!kind_attn || !kind_prefix) return nullptr;
  Py_INCREF(pool);
  Py_XDECREF(workspaces);
  workspaces = pool;
  memcpy(&api, p, sizeof(api));
  Py_RETURN_NONE;
}

// A plain argument: a tensor (or None where allowed), an int or a float.
// `ok` turns false at the first that is not of the accepted form.
struct Args {
  PyObject* const* a;
  bool ok = true;

  const at::Tensor* tensor(int i) {
    if (!THPVariable_CheckExact(a[i])) { ok = false; return nullptr; }
    return &THPVariable_Unpack(a[i]);
  }
  const at::Tensor* maybe(int i) { return a[i] == Py_None ? nullptr : tensor(i); }
  int64_t integer(int i) {
    if (!PyLong_CheckExact(a[i])) { ok = false; return 0; }
    const int64_t v = PyLong_AsLongLong(a[i]);
    if (v == -1 && PyErr_Occurred()) { PyErr_Clear(); ok = false; }
    if (v < INT32_MIN || v > INT32_MAX) ok = false;
    return v;
  }
  double number(int i) {
    if (!PyFloat_CheckExact(a[i])) { ok = false; return 0; }
    return PyFloat_AS_DOUBLE(a[i]);
  }
};

bool dtype_of(const at::Tensor& t, lv_dtype& dt) {
  switch (t.scalar_type()) {
    case at::kFloat: dt = LV_F32; return true;
    case at::kHalf: dt = LV_F16; return true;
    case at::kBFloat16: dt = LV_BF16; return true;
    default: return false;
  }
}

// On `dev`, with real storage (wrapped tensors of transforms have none).
bool on(const at::Tensor* t, const at::Device& dev) {
  return t == nullptr || (t->device() == dev && t->has_storage());
}

bool is_array(const at::Tensor& t, at::ScalarType type, int64_t dim) {
  return t.scalar_type() == type && t.dim() == dim && t.is_contiguous();
}

// [T, >= width] with unit column stride.
bool is_rows(const at::Tensor& t, int64_t width, at::ScalarType type) {
  return t.dim() == 2 && t.size(1) >= width && t.stride(1) == 1 && t.scalar_type() == type;
}

bool is_heads(const at::Tensor& t, int64_t heads, int64_t d) {
  return t.dim() == 3 && t.size(1) == heads && t.size(2) == d && t.stride(2) == 1 &&
         t.stride(1) == d;
}

bool is_cache(const at::Tensor& t) { return t.dim() == 4 && t.is_contiguous(); }

void* ptr(const at::Tensor* t) { return t ? t->data_ptr() : nullptr; }

void* stream_of(const at::Device& dev) { return c10::hip::getCurrentHIPStream(dev.index()).stream(); }

// The wrappers' scratch buffer for (device, stream, kind), if they have made
// one of `bytes` or more (the first call of a size goes through them).
const at::Tensor* scratch(const at::Device& dev, void* stream, size_t bytes, PyObject* kind) {
  PyObject* key = Py_BuildValue("(iKO)", (int)dev.index(), (unsigned long long)(uintptr_t)stream,
                                kind);
  if (!key) { PyErr_Clear(); return nullptr; }
  PyObject* v = PyDict_GetItem(workspaces, key);   // borrowed; no exception set
  Py_DECREF(key);
  if (!v || !THPVariable_CheckExact(v)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(v);
  return (size_t)t.numel() >= bytes ? &t : nullptr;
}

at::Tensor empty(at::IntArrayRef sizes, const at::Tensor& like) {
  return at::empty(sizes, at::TensorOptions().dtype(like.scalar_type()).device(like.device()));
}

bool is_scratch(const at::Tensor& t, size_t bytes) {
  return t.scalar_type() == at::kByte && t.is_contiguous() && (size_t)t.numel() >= bytes;
}

PyObject* done(int rc, const char* what, const at::Tensor* out) {
  if (rc != LV_OK) {
    PyErr_Format(PyExc_RuntimeError, "%s failed (status %d): %s", what, rc, api.last_error());
    return nullptr;
  }
  if (out) return THPVariable_Wrap(*out);
  Py_RETURN_TRUE;
}

#define NOT_PLAIN() Py_RETURN_NONE
#define FAST(NAME, N)                                                               \
  PyObject* NAME##_impl(Args A);                                                    \
  PyObject* NAME(PyObject*, PyObject* const* args, Py_ssize_t n) {                  \
    HANDLE_TH_ERRORS                                                                \
    if (n != N || !api.last_error) {                                                \
      PyErr_Format(PyExc_TypeError, #NAME ": %d arguments of a bound module", N);   \
      return nullptr;                                                               \
    }                                                                               \
    return NAME##_impl(Args{args});                                                 \
    END_HANDLE_TH_ERRORS                                                            \
  }                                                                                 \
  PyObject* NAME##_impl(Args A)

// (key, value, key_cache, value_cache, slot_mapping) -> True
FAST(kv_scatter, 5) {
  const at::Tensor *k = A.tensor(0), *v = A.tensor(1), *kc = A.tensor(2), *vc = A.tensor(3),
                   *slots = A.tensor(4);
  lv_dtype dt;
  if (!A.ok || !kc->is_cuda() || !dtype_of(*kc, dt) || !is_cache(*kc) || !is_cache(*vc) ||
      kc->sizes() != vc->sizes() || vc->scalar_type() != kc->scalar_type())
    NOT_PLAIN();
  const at::Device dev = kc->device();
  const int64_t T = slots->numel(), hkv = kc->size(2), d = kc->size(3);
  if (!on(k, dev) || !on(v, dev) || !on(kc, dev) || !on(vc, dev) || !on(slots, dev) || T == 0 ||
      !is_array(*slots, at::kLong, 1) || !is_heads(*k, hkv, d) || !is_heads(*v, hkv, d) ||
      k->size(0) != T || v->size(0) != T || k->scalar_type() != kc->scalar_type() ||
      v->scalar_type() != kc->scalar_type())
    NOT_PLAIN();
  void* st = stream_of(dev);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = api.kv_scatter(ptr(k), k->stride(0), ptr(v), v->stride(0), ptr(kc), ptr(vc),
                      (const int64_t*)ptr(slots), T, hkv, d, kc->size(1), kc->size(0), dt, st);
  Py_END_ALLOW_THREADS
  return done(rc, "lv_kv_scatter", nullptr);
}

// (query, key_cache, value_cache, block_tables, context_lens, num_kv_heads,
//  scale, cu_seqlens, num_decodes, max_query_len, out, workspace, prefix,
//  prefix_workspace) -> out
FAST(paged_attention, 14) {
  const at::Tensor *q = A.tensor(0), *kc = A.tensor(1), *vc = A.tensor(2), *bt = A.tensor(3),
                   *ctx = A.tensor(4), *cu = A.maybe(7), *given = A.maybe(10), *ws = A.maybe(11);
  const double scale = A.number(6);
  const int64_t max_q = A.integer(9);
  lv_dtype dt;
  if (!A.ok || !kc->is_cuda() || !dtype_of(*q, dt) || q->dim() != 3) NOT_PLAIN();
  const at::Device dev = kc->device();
  const int64_t T = q->size(0), H = q->size(1), D = q->size(2);
  if (!on(q, dev) || !on(kc, dev) || !on(vc, dev) || !on(bt, dev) || !on(ctx, dev) ||
      !on(cu, dev) || !on(given, dev) || !on(ws, dev) || !is_heads(*q, H, D) || !is_cache(*kc) ||
      !is_cache(*vc) || kc->sizes() != vc->sizes() || kc->size(3) != D ||
      kc->scalar_type() != q->scalar_type() || vc->scalar_type() != q->scalar_type() ||
      !is_array(*bt, at::kInt, 2) || !is_array(*ctx, at::kInt, 1))
    NOT_PLAIN();
  const int64_t n_blocks = kc->size(0), bs = kc->size(1), hkv = kc->size(2), B = bt->size(0),
                max_blocks = bt->size(1);
  if (A.a[5] != Py_None && A.integer(5) != hkv) NOT_PLAIN();
  int64_t nd = cu ? 0 : B;
  if (A.a[8] != Py_None) nd = A.integer(8);
  if (!A.ok || B == 0 || ctx->size(0) != B || nd < 0 || nd > B ||
      (cu ? !is_array(*cu, at::kInt, 1) || cu->size(0) != B + 1 : T != B) ||
      max_blocks > INT32_MAX || T > INT32_MAX)
    NOT_PLAIN();
  if (given && (!is_heads(*given, H, D) || given->size(0) != T ||
                given->scalar_type() != q->scalar_type()))
    NOT_PLAIN();
  size_t ws_bytes = api.attention_ws(B, nd, T, H, D, bs, max_blocks, max_q, dt);
  if (ws && !is_scratch(*ws, ws_bytes)) NOT_PLAIN();
  // shared prefixes: PrefixPlan(blocks, items, members)
  const at::Tensor *pb = nullptr, *pi = nullptr, *pm = nullptr, *pws = nullptr;
  size_t pws_bytes = 0;
  if (A.a[12] != Py_None) {
    if (!PyTuple_Check(A.a[12]) || PyTuple_GET_SIZE(A.a[12]) != 3) NOT_PLAIN();
    Args P{((PyTupleObject*)A.a[12])->ob_item};
    pb = P.tensor(0); pi = P.tensor(1); pm = P.tensor(2);
    pws = A.maybe(13);
    pws_bytes = api.prefix_ws(nd, H, D);
    if (!P.ok || !A.ok || !on(pb, dev) || !on(pi, dev) || !on(pm, dev) || !on(pws, dev) ||
        !is_array(*pb, at::kInt, 1) || !is_array(*pi, at::kInt, 2) ||
        !is_array(*pm, at::kInt, 1) || pb->size(0) != nd || pi->size(1) != 4 ||
        (pws && !is_scratch(*pws, pws_bytes)))
      NOT_PLAIN();
  }
  void* st = stream_of(dev);
  if (!ws && nd < B &&
      c10::hip::currentStreamCaptureStatusMayInitCtx() == c10::hip::CaptureStatus::None)
    ws_bytes = api.split_ws(B, nd, T, H, hkv, D, bs, max_blocks, max_q, dt);
  if (ws) ws_bytes = ws->numel();
  else if (ws_bytes > 0 && !(ws = scratch(dev, st, ws_bytes, kind_attn))) NOT_PLAIN();
  if (pb && !pws && pws_bytes > 0 && !(pws = scratch(dev, st, pws_bytes, kind_prefix)))
    NOT_PLAIN();
  // held past the GIL's release: another thread may grow the pool's entry
  const at::Tensor ws_held = ws ? *ws : at::Tensor(), pws_held = pws ? *pws : at::Tensor();
  const at::Tensor out = given ? *given : empty(q->sizes(), *q);
  void *wp = ptr(ws), *pwp = ptr(pws);
  const size_t pwn = pws ? pws->numel() : 0;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  if (pb)
    rc = api.attention_prefix(ptr(q), q->stride(0), ptr(kc), ptr(vc), n_blocks,
                              (const int32_t*)ptr(bt), max_blocks, (const int32_t*)ptr(cu),
                              (const int32_t*)ptr(ctx), B, nd, T, max_q, H, hkv, D, bs,
                              (float)scale, out.data_ptr(), out.stride(0), wp, ws_bytes,
                              (const int32_t*)ptr(pb), (const int32_t*)ptr(pi), pi->size(0),
                              (const int32_t*)ptr(pm), pm->size(0), pwp, pwn, dt, st);
  else
    rc = api.attention(ptr(q), q->stride(0), ptr(kc), ptr(vc), n_blocks, (const int32_t*)ptr(bt),
                       max_blocks, (const int32_t*)ptr(cu), (const int32_t*)ptr(ctx), B, nd, T,
                       max_q, H, hkv, D, bs, (float)scale, out.data_ptr(), out.stride(0), wp,
                       ws_bytes, dt, st);
  Py_END_ALLOW_THREADS
  return done(rc, pb ? "lv_paged_attention_prefix" : "lv_paged_attention", &out);
}

// (logits, temperature, uniform, out, workspace) -> out
FAST(sample, 5) {
  const at::Tensor *x = A.tensor(0), *temp = A.tensor(1), *uni = A.tensor(2), *given = A.maybe(3),
                   *ws = A.maybe(4);
  lv_dtype dt;
  if (!A.ok || !x->is_cuda() || !dtype_of(*x, dt) || x->dim() != 2 || x->stride(1) != 1)
    NOT_PLAIN();
  const at::Device dev = x->device();
  const int64_t B = x->size(0), V = x->size(1);
  if (B == 0 || !on(x, dev) || !on(temp, dev) || !on(uni, dev) || !on(given, dev) ||
      !on(ws, dev) || !is_array(*temp, at::kFloat, 1) || temp->size(0) != B ||
      !is_array(*uni, at::kFloat, 1) || uni->size(0) != B ||
      (given && (!is_array(*given, at::kLong, 1) || given->size(0) != B)))
    NOT_PLAIN();
  const size_t bytes = api.sample_ws(B, V);
  if (bytes == 0 || (ws && !is_scratch(*ws, bytes))) NOT_PLAIN();
  void* st = stream_of(dev);
  if (!ws && !(ws = scratch(dev, st, bytes, kind_attn))) NOT_PLAIN();
  const at::Tensor ws_held = *ws;   // another thread may grow the pool's entry
  const at::Tensor out =
      given ? *given : at::empty({B}, at::TensorOptions().dtype(at::kLong).device(dev));
  void* wp = ptr(ws);
  const size_t wn = ws->numel();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = api.sample(ptr(x), B, V, x->stride(0), (const float*)ptr(temp), (const float*)ptr(uni),
                  (int64_t*)out.data_ptr(), wp, wn, dt, st);
  Py_END_ALLOW_THREADS
  return done(rc, "lv_sample", &out);
}

// (x, weight, eps, residual, out) -> out
FAST(add_rms_norm, 5) {
  const at::Tensor *x = A.tensor(0), *w = A.tensor(1), *res = A.maybe(3), *given = A.maybe(4);
  const double eps = A.number(2);
  lv_dtype dt;
  if (!A.ok || !x->is_cuda() || !dtype_of(*x, dt) || x->dim() != 2) NOT_PLAIN();
  const at::Device dev = x->device();
  const int64_t T = x->size(0), hidden = x->size(1);
  const at::ScalarType type = x->scalar_type();
  if (T == 0 || !on(x, dev) || !on(w, dev) || !on(res, dev) || !on(given, dev) ||
      !is_rows(*x, hidden, type) || !is_array(*w, type, 1) || w->size(0) != hidden ||
      (res && (!is_rows(*res, hidden, type) || res->size(0) != T)) ||
      (given && (!is_rows(*given, hidden, type) || given->size(0) != T)))
    NOT_PLAIN();
  const at::Tensor out = given ? *given : empty({T, hidden}, *x);
  void* st = stream_of(dev);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = api.add_rms_norm(ptr(x), x->stride(0), ptr(res), res ? res->stride(0) : 0, ptr(w),
                        out.data_ptr(), out.stride(0), T, hidden, (float)eps, dt, st);
  Py_END_ALLOW_THREADS
  return done(rc, "lv_add_rms_norm", &out);
}

// (qkv, num_heads, num_kv_heads, head_dim, cos, sin, positions, slot_mapping,
//  key_cache, value_cache, q_norm_weight, k_norm_weight, eps, q_out) -> q_out
FAST(qk_norm_rope_cache, 14) {
  const at::Tensor *qkv = A.tensor(0), *cs = A.tensor(4), *sn = A.tensor(5), *pos = A.tensor(6),
                   *slots = A.tensor(7), *kc = A.tensor(8), *vc = A.tensor(9), *qw = A.maybe(10),
                   *kw = A.maybe(11), *given = A.maybe(13);
  const int64_t H = A.integer(1), Hkv = A.integer(2), D = A.integer(3);
  const double eps = A.number(12);
  lv_dtype dt;
  if (!A.ok || H < 1 || Hkv < 1 || D < 1 || !qkv->is_cuda() || !dtype_of(*qkv, dt)) NOT_PLAIN();
  const at::Device dev = qkv->device();
  const at::ScalarType type = qkv->scalar_type();
  for (const at::Tensor* t : {qkv, cs, sn, pos, slots, kc, vc, qw, kw, given})
    if (!on(t, dev)) NOT_PLAIN();
  if (!is_rows(*qkv, (H + 2 * Hkv) * D, type) || !is_array(*pos, at::kLong, 1) ||
      !is_array(*slots, at::kLong, 1))
    NOT_PLAIN();
  const int64_t T = qkv->size(0);
  if (T == 0 || pos->size(0) != T || slots->size(0) != T || !is_cache(*kc) || !is_cache(*vc) ||
      kc->scalar_type() != type || vc->scalar_type() != type || kc->sizes() != vc->sizes() ||
      kc->size(2) != Hkv || kc->size(3) != D)
    NOT_PLAIN();
  for (const at::Tensor* t : {cs, sn})
    if (!is_array(*t, type, 2) || t->size(1) != D / 2) NOT_PLAIN();
  if (sn->size(0) < cs->size(0)) NOT_PLAIN();
  for (const at::Tensor* t : {qw, kw})
    if (t && (!is_array(*t, type, 1) || t->size(0) != D)) NOT_PLAIN();
  if (given && (!is_heads(*given, H, D) || given->size(0) != T || given->scalar_type() != type))
    NOT_PLAIN();
  const at::Tensor out = given ? *given : empty({T, H, D}, *qkv);
  void* st = stream_of(dev);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = api.qk_norm_rope_cache(ptr(qkv), qkv->stride(0), ptr(qw), ptr(kw), ptr(cs), ptr(sn),
                              cs->size(0), (const int64_t*)ptr(pos), (const int64_t*)ptr(slots),
                              out.data_ptr(), out.stride(0), ptr(kc), ptr(vc), kc->size(0),
                              kc->size(1), T, H, Hkv, D, (float)eps, dt, st);
  Py_END_ALLOW_THREADS
  return done(rc, "lv_qk_norm_rope_cache", &out);
}

// (gate_up, out) -> out
FAST(silu_mul, 2) {
  const at::Tensor *x = A.tensor(0), *given = A.maybe(1);
  lv_dtype dt;
  if (!A.ok || !x->is_cuda() || !dtype_of(*x, dt) || x->dim() != 2) NOT_PLAIN();
  const at::Device dev = x->device();
  const int64_t T = x->size(0), inter = x->size(1) / 2;
  if (T == 0 || !on(x, dev) || !on(given, dev) || !is_rows(*x, 2 * inter, x->scalar_type()) ||
      (given && (!is_rows(*given, inter, x->scalar_type()) || given->size(0) != T)))
    NOT_PLAIN();
  const at::Tensor out = given ? *given : empty({T, inter}, *x);
  void* st = stream_of(dev);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = api.silu_mul(ptr(x), x->stride(0), out.data_ptr(), out.stride(0), T, inter, dt, st);
  Py_END_ALLOW_THREADS
  return done(rc, "lv_silu_mul", &out);
}

// (x, weight, silu_mul, out) -> out
FAST(linear, 4) {
  const at::Tensor *x = A.tensor(0), *w = A.tensor(1), *given = A.maybe(3);
  const int64_t act = A.integer(2);
  lv_dtype dt;
  if (!A.ok || !x->is_cuda() || !dtype_of(*x, dt) || x->dim() != 2 || w->dim() != 2) NOT_PLAIN();
  const at::Device dev = x->device();
  const at::ScalarType type = x->scalar_type();
  const int64_t M = x->size(0), K = x->size(1), rows = w->size(0);
  const int64_t N = act == LV_ACT_SILU_MUL ? rows / 2 : rows;
  if (M == 0 || !on(x, dev) || !on(w, dev) || !on(given, dev) || !is_rows(*x, K, type) ||
      !is_rows(*w, K, type) || w->size(1) != K || (act == LV_ACT_SILU_MUL && rows % 2) ||
      (given && (!is_rows(*given, N, type) || given->size(0) != M)))
    NOT_PLAIN();
  const at::Tensor out = given ? *given : empty({M, N}, *x);
  void* st = stream_of(dev);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = api.linear(ptr(x), x->stride(0), ptr(w), w->stride(0), out.data_ptr(), out.stride(0), M, N,
                  K, act, dt, st);
  Py_END_ALLOW_THREADS
  return done(rc, "lv_linear", &out);
}

// (x, weight, out) -> out
FAST(linear_f32, 3) {
  const at::Tensor *x = A.tensor(0), *w = A.tensor(1), *given = A.maybe(2);
  if (!A.ok || !x->is_cuda() || x->scalar_type() != at::kFloat || x->dim() != 2 || w->dim() != 2)
    NOT_PLAIN();
  const at::Device dev = x->device();
  const int64_t M = x->size(0), K = x->size(1), N = w->size(0);
  if (M == 0 || !on(x, dev) || !on(w, dev) || !on(given, dev) || !is_rows(*x, K, at::kFloat) ||
      !is_rows(*w, K, at::kFloat) || w->size(1) != K ||
      (given && (!is_rows(*given, N, at::kFloat) || given->size(0) != M)))
    NOT_PLAIN();
  const at::Tensor out = given ? *given : empty({M, N}, *x);
  void* st = stream_of(dev);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = api.linear_f32((const float*)ptr(x), x->stride(0), (const float*)ptr(w), w->stride(0),
                      (float*)out.data_ptr(), out.stride(0), M, N, K, st);
  Py_END_ALLOW_THREADS
  return done(rc, "lv_linear_f32", &out);
}

// No tangent of forward-mode differentiation, and nothing between the tensor
// and the values in its storage: no transform's wrapper, lazy conjugate or
// negation.
bool is_direct(const at::Tensor& t) {
  using K = at::DispatchKey;
  static const uint64_t plain =
      at::DispatchKeySet({K::CUDA, K::AutogradCUDA, K::AutocastCUDA, K::ADInplaceOrView}).raw_repr();
  return (t.key_set().raw_repr() & ~plain) == 0 && !t._fw_grad(/*level=*/0).defined();
}

// This thread's layers leave their products to nn.Linear (library_products).
thread_local bool products_by_library = false;

// Nobody but the dispatcher's CUDA kernel would see a call made now: neither
// autograd, autocast, a trace, a transform nor a Python mode.
bool calls_are_direct() {
  if (products_by_library || at::GradMode::is_enabled() || at::autocast::is_autocast_enabled(at::kCUDA) ||
      at::impl::torch_function_mode_enabled() ||
      c10::impl::TorchDispatchModeTLS::any_modes_set())
    return false;
  const auto tls = c10::impl::tls_local_dispatch_key_set();
  return (tls.included_.raw_repr() & ~c10::default_included_set.raw_repr()) == 0;
}

// Rows of `width` elements, each on a 16-byte boundary and none overlapping
// the next.
bool is_aligned_rows(const at::Tensor& t, int64_t width, at::ScalarType type) {
  return is_rows(t, width, type) && t.stride(0) >= width &&
         t.stride(0) * t.element_size() % 16 == 0 && (uintptr_t)ptr(&t) % 16 == 0;
}

// (x, weight, None or "silu_mul") -> out: nn.Linear's product for a layer that
// falls back on nn.Linear itself, so everything the library's kernels ask for
// or nn.Linear answers differently is not plain here.  What these products save
// is host time; on the GPU the library GEMM is often the faster (fp32, 16 rows
// of 1024x512: 7.2 us against 4.5; 4096x1024 11.9 and 6.0), so the decode graphs
// switch them off (library_products).  That a stream is capturing does not: the
// warm-up before a capture has to take the capture's route, or the library's
// handle for the thread would be made inside it, which the runtime does not
// survive.  bf16 / fp16, 257-512 rows, GPU time against the
// library: 0.65-1.13 where the workgroups run at once and k is at least 512
// (4096x1024 1.01-1.10, 1024x3072 0.83-0.91), 1.2-1.7 where they do not
// (6144x1024 from 384 rows on, 2048x2048 up to 384, 384 rows of 1280x5120); with
// SiLU 0.64-0.85 where the layer widens, up to 1.35 where it does not.
FAST(layer_linear, 3) {
  const at::Tensor *x = A.tensor(0), *w = A.tensor(1);
  const bool silu = A.a[2] != Py_None;
  lv_dtype dt;
  if (!A.ok || !x->is_cuda() || !dtype_of(*x, dt) || x->dim() != 2 || w->dim() != 2 ||
      (silu && (!PyUnicode_Check(A.a[2]) ||
                PyUnicode_CompareWithASCIIString(A.a[2], "silu_mul") != 0)) ||
      !calls_are_direct())
    NOT_PLAIN();
  const at::Device dev = x->device();
  const at::ScalarType type = x->scalar_type();
  const int64_t M = x->size(0), K = x->size(1), rows = w->size(0);
  const int64_t N = silu ? rows / 2 : rows;
  const int32_t act = silu ? LV_ACT_SILU_MUL : LV_ACT_NONE;
  if (M == 0 || N == 0 || K == 0 || !on(x, dev) || !on(w, dev) || !is_direct(*x) ||
      !is_direct(*w) || w->size(1) != K || (silu && rows % 2) || !is_aligned_rows(*x, K, type) ||
      !is_aligned_rows(*w, K, type) ||
      (dt == LV_F32 ? silu || K % 4 != 0
                    : (silu ? N < K : K < 512) || !api.linear_one_round(M, N, K, act)))
    NOT_PLAIN();
  const at::Tensor out = empty({M, N}, *x);
  void* st = stream_of(dev);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  if (dt == LV_F32)
    rc = api.linear_f32((const float*)ptr(x), x->stride(0), (const float*)ptr(w), w->stride(0),
                        (float*)out.data_ptr(), out.stride(0), M, N, K, st);
  else
    rc = api.linear(ptr(x), x->stride(0), ptr(w), w->stride(0), out.data_ptr(), out.stride(0), M,
                    N, K, act, dt, st);
  Py_END_ALLOW_THREADS
  return done(rc, dt == LV_F32 ? "lv_linear_f32" : "lv_linear", &out);
}

// (on) -> whether it was: layer_linear answers None to this thread from here on.
PyObject* library_products(PyObject*, PyObject* on) {
  const int v = PyObject_IsTrue(on);
  if (v < 0) return nullptr;
  const bool was = products_by_library;
  products_by_library = v != 0;
  return PyBool_FromLong(was);
}

#define METHOD(NAME) {#NAME, (PyCFunction)(void (*)(void))NAME, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {{"bind", bind, METH_VARARGS, nullptr},
                         {"library_products", library_products, METH_O, nullptr},
                         METHOD(kv_scatter),
                         METHOD(paged_attention),
                         METHOD(sample),
                         METHOD(add_rms_norm),
                         METHOD(qk_norm_rope_cache),
                         METHOD(silu_mul),
                         METHOD(linear),
                         METHOD(linear_f32),
                         METHOD(layer_linear),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module); }
