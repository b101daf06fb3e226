// Native fast path of ops.py (CPython extension module _native).
//
// Each function takes its op's arguments in order, checks them, allocates the
// output through torch and calls libmce.so on torch's current stream.  It
// handles the plain case -- ordinary GPU tensors (no subclass, no functorch or
// other wrapper) whose types, shapes and layouts the kernels take as they are
// -- and otherwise returns NotImplemented with nothing done: ops.py then runs
// its own checks, copies and error reports.  A call that the library refuses
// (before any launch) also returns NotImplemented, so that ops.py repeats it
// and reports the error.
//
// What it is for: the same steps in Python took 8.7 (rmsnorm) to 17 us (fused
// RoPE + KV store) a call on the host, longer than the kernels of a decode
// batch or a short prompt.  The library's entry points are handed over once
// as addresses by _lib.load() (bind), after its ABI version check.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <exception>

#include "mce_abi.h"
#include "mce_internal.h"

namespace {

// ---- the library's entry points ------------------------------------------
#define MCE_NATIVE_ENTRIES(X)                                                              \
  X(mce_rmsnorm)                                                                           \
  X(mce_swiglu)                                                                            \
  X(mce_paged_kv_store)                                                                    \
  X(mce_rope_inplace)                                                                      \
  X(mce_rope_kv_store)                                                                     \
  X(mce_paged_attention_decode_workspace_size)                                             \
  X(mce_paged_attention_decode)                                                            \
  X(mce_paged_attention_decode_rope)                                                       \
  X(mce_prefill_attention_strided)                                                         \
  X(mce_prefill_attention_paged_workspace_size)                                            \
  X(mce_prefill_attention_paged)                                                           \
  X(mce_decode_gemm)                                                                       \
  X(mce_rmsnorm_decode_gemm)                                                               \
  X(mce_prompt_gemm_takes)                                                                 \
  X(mce_prompt_gemm_workspace_size)                                                        \
  X(mce_prompt_gemm)
struct Entries {
#define X(name) decltype(&::name) name = nullptr;
  MCE_NATIVE_ENTRIES(X)
#undef X
};
Entries g_lib;
bool g_bound = false;  // written with the GIL held, before any use

// ---- arguments -------------------------------------------------------------
// A plain tensor on a GPU: what data_ptr(), sizes and strides say is all there
// is to it.
const at::Tensor *plain(PyObject *o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor &t = THPVariable_Unpack(o);
  using K = c10::DispatchKey;
  static const c10::DispatchKeySet wrapped{
      K::Python,         K::PythonTLSSnapshot,     K::FuncTorchBatched, K::FuncTorchGradWrapper,
      K::Functionalize,  K::Conjugate,             K::Negative,         K::ZeroTensor,
      K::Batched,        K::FuncTorchDynamicLayerBackMode};
  if (!t.defined() || !t.is_cuda() || t.layout() != c10::kStrided || t.key_set().has_any(wrapped) ||
      !t.has_storage())
    return nullptr;
  return &t;
}

int dtype_code(const at::Tensor &t) {
  return t.scalar_type() == at::kHalf ? MCE_F16 : t.scalar_type() == at::kBFloat16 ? MCE_BF16 : -1;
}

bool as_int(PyObject *o, int64_t *out) {
  if (!PyLong_CheckExact(o)) return false;
  int over = 0;
  *out = PyLong_AsLongLongAndOverflow(o, &over);
  return over == 0 && !(*out == -1 && PyErr_Occurred());
}
bool as_float(PyObject *o, float *out) {
  if (!PyFloat_CheckExact(o)) return false;
  *out = (float)PyFloat_AS_DOUBLE(o);
  return true;
}

// contiguous int32 of n elements on dev
bool ints(const at::Tensor *t, int64_t n, c10::Device dev) {
  return t && t->scalar_type() == at::kInt && t->numel() == n && t->is_contiguous() && t->device() == dev;
}
// contiguous fp32 [P, d / 2] cos and sin tables on dev
bool tables(const at::Tensor *c, const at::Tensor *s, int64_t d, c10::Device dev) {
  if (!c || !s) return false;
  for (const at::Tensor *t : {c, s})
    if (t->scalar_type() != at::kFloat || t->dim() != 2 || t->size(1) != d / 2 ||
        !t->is_contiguous() || t->device() != dev)
      return false;
  return c->size(0) == s->size(0);
}
// contiguous [num_blocks, block_size, heads, d] pools like ref
bool pools(const at::Tensor *k, const at::Tensor *v, const at::Tensor &ref, int64_t heads, int64_t d) {
  if (!k || !v) return false;
  for (const at::Tensor *t : {k, v})
    if (t->scalar_type() != ref.scalar_type() || t->device() != ref.device() || t->dim() != 4 ||
        !t->is_contiguous())
      return false;
  return k->sizes() == v->sizes() && (heads < 0 || k->size(2) == heads) && k->size(3) == d;
}
bool fits_int(std::initializer_list<int64_t> v) {
  for (int64_t x : v)
    if (x < 0 || x > INT32_MAX) return false;
  return true;
}

PyObject *declined() { Py_RETURN_NOTIMPLEMENTED; }

void *stream_of(c10::Device dev) {
  return (void *)c10::hip::getCurrentHIPStream(dev.index()).stream();
}

// A 256-byte aligned workspace from torch's allocator, ordered with the
// current stream like any other temporary.
struct Workspace {
  at::Tensor t;
  void *ptr = nullptr;
  Workspace(size_t bytes, const at::Tensor &like) {
    if (bytes == 0) return;
    t = at::empty({(int64_t)bytes + 256}, like.options().dtype(at::kByte));
    ptr = (void *)(((uintptr_t)t.data_ptr() + 255) & ~(uintptr_t)255);
  }
};

// Calls the library without the GIL.
template <class F>
int launch(F &&f) {
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = f();
  Py_END_ALLOW_THREADS
  return rc;
}

PyObject *result(int rc, const at::Tensor &out) {
  return rc == MCE_OK ? THPVariable_Wrap(out) : declined();
}
PyObject *done(int rc) {
  if (rc != MCE_OK) return declined();
  Py_RETURN_NONE;
}

// ---- the ops ---------------------------------------------------------------
PyObject *rmsnorm(PyObject *const *a) {
  const at::Tensor *x = plain(a[0]), *w = plain(a[1]);
  float eps;
  if (!x || !w || !as_float(a[2], &eps)) return declined();
  const int code = dtype_code(*x);
  if (code < 0 || w->scalar_type() != x->scalar_type() || w->device() != x->device() ||
      x->dim() < 1 || !x->is_contiguous())
    return declined();
  const int64_t h = x->size(-1);
  if (h < 1 || w->dim() != 1 || w->size(0) != h || !w->is_contiguous()) return declined();
  const c10::DeviceGuard guard(x->device());
  at::Tensor out = at::empty_like(*x);
  const void *xp = x->data_ptr(), *wp = w->data_ptr();
  void *op = out.data_ptr(), *st = stream_of(x->device());
  const int64_t rows = x->numel() / h;
  return result(launch([&] { return g_lib.mce_rmsnorm(code, xp, wp, op, rows, h, h, h, eps, st); }), out);
}

PyObject *swiglu(PyObject *const *a) {
  const at::Tensor *x = plain(a[0]);
  if (!x) return declined();
  const int code = dtype_code(*x);
  if (code < 0 || x->dim() < 1 || !x->is_contiguous()) return declined();
  const int64_t w = x->size(-1);
  if (w < 2 || w % 2 != 0) return declined();
  const c10::DeviceGuard guard(x->device());
  c10::SmallVector<int64_t, 5> shape(x->sizes().begin(), x->sizes().end());
  shape.back() = w / 2;
  at::Tensor out = at::empty(shape, x->options());
  const void *xp = x->data_ptr();
  void *op = out.data_ptr(), *st = stream_of(x->device());
  const int64_t rows = x->numel() / w;
  return result(launch([&] { return g_lib.mce_swiglu(code, xp, op, rows, w / 2, w, w / 2, st); }), out);
}

PyObject *paged_kv_store(PyObject *const *a) {
  const at::Tensor *k = plain(a[0]), *v = plain(a[1]), *kc = plain(a[2]), *vc = plain(a[3]),
                   *sm = plain(a[4]);
  if (!k || !v || k->dim() != 3) return declined();
  const int code = dtype_code(*k);
  const int64_t n = k->size(0), h = k->size(1), d = k->size(2);
  if (code < 0 || v->scalar_type() != k->scalar_type() || v->device() != k->device() ||
      v->sizes() != k->sizes() || !pools(kc, vc, *k, h, d) || k->stride(2) != 1 || v->stride(2) != 1 ||
      !ints(sm, n, k->device()) || sm->dim() != 1 || !fits_int({h, d, kc->size(1)}))
    return declined();
  const c10::DeviceGuard guard(k->device());
  const void *kp = k->data_ptr(), *vp = v->data_ptr();
  void *kcp = kc->data_ptr(), *vcp = vc->data_ptr(), *st = stream_of(k->device());
  const int32_t *sp = (const int32_t *)sm->data_ptr();
  const int64_t ks0 = k->stride(0), ks1 = k->stride(1), vs0 = v->stride(0), vs1 = v->stride(1);
  const int64_t nb = kc->size(0);
  const int bs = (int)kc->size(1);
  return done(launch([&] {
    return g_lib.mce_paged_kv_store(code, kp, vp, kcp, vcp, sp, n, (int)h, (int)d, bs, nb, ks0, ks1,
                                    vs0, vs1, st);
  }));
}

PyObject *paged_attention_decode(PyObject *const *a) {
  const at::Tensor *q = plain(a[0]), *kc = plain(a[1]), *vc = plain(a[2]), *bt = plain(a[3]),
                   *cl = plain(a[4]);
  int64_t mb, bs;
  float scale;
  if (!q || !as_int(a[5], &mb) || !as_int(a[6], &bs) || !as_float(a[7], &scale)) return declined();
  const int code = dtype_code(*q);
  if (code < 0 || q->dim() != 3 || !q->is_contiguous()) return declined();
  const int64_t b = q->size(0), hq = q->size(1), d = q->size(2);
  if (!pools(kc, vc, *q, -1, d) || bs != kc->size(1) || b < 1 || !ints(bt, b * mb, q->device()) ||
      bt->dim() != 2 || bt->size(1) != mb || !ints(cl, b, q->device()) || cl->dim() != 1 ||
      !fits_int({b, hq, d, mb, bs, kc->size(2)}))
    return declined();
  const int hkv = (int)kc->size(2);
  const c10::DeviceGuard guard(q->device());
  at::Tensor out = at::empty_like(*q);
  const size_t ws_bytes =
      g_lib.mce_paged_attention_decode_workspace_size((int)b, (int)hq, hkv, (int)mb, (int)bs);
  const Workspace ws(ws_bytes, *q);
  const void *qp = q->data_ptr(), *kp = kc->data_ptr(), *vp = vc->data_ptr();
  const int32_t *bp = (const int32_t *)bt->data_ptr(), *cp = (const int32_t *)cl->data_ptr();
  void *op = out.data_ptr(), *st = stream_of(q->device());
  const int64_t nb = kc->size(0);
  return result(launch([&] {
                  return g_lib.mce_paged_attention_decode(code, qp, kp, vp, bp, cp, op, (int)b, (int)hq,
                                                          hkv, (int)d, (int)mb, (int)bs, nb, scale,
                                                          ws.ptr, ws_bytes, st);
                }),
                out);
}

PyObject *rope_inplace(PyObject *const *a) {
  const at::Tensor *q = plain(a[0]), *k = a[1] == Py_None ? nullptr : plain(a[1]),
                   *c = plain(a[2]), *s = plain(a[3]), *pos = plain(a[4]);
  if (!q || q->dim() != 4 || (a[1] != Py_None && !k)) return declined();
  const int code = dtype_code(*q);
  const int64_t b = q->size(0), n = q->size(1), hq = q->size(2), d = q->size(3);
  if (code < 0 || d % 2 != 0 || q->stride(3) != 1 || !tables(c, s, d, q->device()) ||
      !ints(pos, b * n, q->device()))
    return declined();
  if (k && (k->scalar_type() != q->scalar_type() || k->device() != q->device() || k->dim() != 4 ||
            k->size(0) != b || k->size(1) != n || k->size(3) != d || k->stride(3) != 1))
    return declined();
  const int64_t hkv = k ? k->size(2) : 0;
  if (!fits_int({b, n, hq, hkv, d})) return declined();
  const c10::DeviceGuard guard(q->device());
  void *qp = q->data_ptr(), *kp = k ? k->data_ptr() : nullptr, *st = stream_of(q->device());
  const float *cp = (const float *)c->data_ptr(), *sp = (const float *)s->data_ptr();
  const int32_t *pp = (const int32_t *)pos->data_ptr();
  const int64_t rows = c->size(0), q0 = q->stride(0), q1 = q->stride(1), q2 = q->stride(2);
  const int64_t k0 = k ? k->stride(0) : 0, k1 = k ? k->stride(1) : 0, k2 = k ? k->stride(2) : 0;
  return done(launch([&] {
    return g_lib.mce_rope_inplace(code, qp, kp, cp, sp, pp, (int)b, (int)n, (int)hq, (int)hkv, (int)d,
                                  rows, q0, q1, q2, k0, k1, k2, st);
  }));
}

PyObject *rope_kv_store(PyObject *const *a) {
  const at::Tensor *q = plain(a[0]), *k = plain(a[1]), *v = plain(a[2]), *kc = plain(a[3]),
                   *vc = plain(a[4]), *c = plain(a[5]), *s = plain(a[6]), *pos = plain(a[7]),
                   *sm = plain(a[8]), *qo = a[9] == Py_None ? nullptr : plain(a[9]);
  if (!q || !k || !v || (a[9] != Py_None && !qo) || q->dim() != 3 || k->dim() != 3) return declined();
  const int code = dtype_code(*q);
  const int64_t n = q->size(0), hq = q->size(1), d = q->size(2), hkv = k->size(1);
  const c10::Device dev = q->device();
  if (code < 0 || k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type() ||
      k->device() != dev || v->device() != dev || v->sizes() != k->sizes() || k->size(0) != n ||
      k->size(2) != d || d % 2 != 0 || q->stride(2) != 1 || k->stride(2) != 1 || v->stride(2) != 1 ||
      !pools(kc, vc, *q, hkv, d) || !tables(c, s, d, dev) || !ints(pos, n, dev) || !ints(sm, n, dev) ||
      !fits_int({hq, hkv, d, kc->size(1)}))
    return declined();
  if (qo && (qo->scalar_type() != q->scalar_type() || qo->sizes() != q->sizes() ||
             !qo->is_contiguous() || qo->device() != dev))
    return declined();
  // the one-launch layouts only: the library runs others as two operations in
  // place, which must not be repeated after an error between them
  for (const at::Tensor *t : {q, k, v, kc, vc, c, s, qo})
    if (t && (uintptr_t)t->data_ptr() % 16 != 0) return declined();
  for (const at::Tensor *t : {q, k, v})
    if (d % 8 != 0 || t->stride(0) % 8 != 0 || t->stride(1) % 8 != 0) return declined();
  const c10::DeviceGuard guard(dev);
  void *qp = q->data_ptr(), *qop = qo ? qo->data_ptr() : nullptr, *kp = k->data_ptr();
  const void *vp = v->data_ptr();
  void *kcp = kc->data_ptr(), *vcp = vc->data_ptr(), *st = stream_of(dev);
  const float *cp = (const float *)c->data_ptr(), *sp = (const float *)s->data_ptr();
  const int32_t *pp = (const int32_t *)pos->data_ptr(), *smp = (const int32_t *)sm->data_ptr();
  const int64_t rows = c->size(0), nb = kc->size(0);
  const int bs = (int)kc->size(1);
  const int64_t q0 = q->stride(0), q1 = q->stride(1), k0 = k->stride(0), k1 = k->stride(1),
                v0 = v->stride(0), v1 = v->stride(1);
  return done(launch([&] {
    return g_lib.mce_rope_kv_store(code, qp, qop, kp, vp, kcp, vcp, cp, sp, pp, smp, n, (int)hq,
                                   (int)hkv, (int)d, rows, bs, nb, q0, q1, k0, k1, v0, v1, st);
  }));
}

PyObject *decode_rope_attention(PyObject *const *a) {
  const at::Tensor *q = plain(a[0]), *k = plain(a[1]), *v = plain(a[2]), *kc = plain(a[3]),
                   *vc = plain(a[4]), *c = plain(a[5]), *s = plain(a[6]), *pos = plain(a[7]),
                   *sm = plain(a[8]), *bt = plain(a[9]), *cl = plain(a[10]);
  int64_t mb;
  float scale;
  if (!q || !k || !v || !as_int(a[11], &mb) || !as_float(a[12], &scale) || q->dim() != 3 ||
      k->dim() != 3)
    return declined();
  const int code = dtype_code(*q);
  const int64_t b = q->size(0), hq = q->size(1), d = q->size(2), hkv = k->size(1);
  const c10::Device dev = q->device();
  if (code < 0 || k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type() ||
      k->device() != dev || v->device() != dev || v->sizes() != k->sizes() || k->size(0) != b ||
      k->size(2) != d || !pools(kc, vc, *q, hkv, d) || !tables(c, s, d, dev) || !ints(pos, b, dev) ||
      !ints(sm, b, dev) || !ints(cl, b, dev) || !ints(bt, b * mb, dev) || bt->dim() != 2 ||
      bt->size(1) != mb || k->stride(0) != v->stride(0) ||
      !fits_int({b, hq, hkv, d, mb, kc->size(1), mb * kc->size(1)}))
    return declined();
  for (const at::Tensor *t : {q, k, v})
    if (t->stride(2) != 1 || t->stride(1) != d) return declined();
  const c10::DeviceGuard guard(dev);
  at::Tensor out = at::empty({b, hq, d}, q->options());
  const void *qp = q->data_ptr(), *kp = k->data_ptr(), *vp = v->data_ptr();
  void *kcp = kc->data_ptr(), *vcp = vc->data_ptr(), *op = out.data_ptr(), *st = stream_of(dev);
  const float *cp = (const float *)c->data_ptr(), *sp = (const float *)s->data_ptr();
  const int32_t *pp = (const int32_t *)pos->data_ptr(), *smp = (const int32_t *)sm->data_ptr(),
                *bp = (const int32_t *)bt->data_ptr(), *clp = (const int32_t *)cl->data_ptr();
  const int64_t rows = c->size(0), nb = kc->size(0), qs = q->stride(0), ks = k->stride(0);
  const int bs = (int)kc->size(1);
  return result(launch([&] {
                  return g_lib.mce_paged_attention_decode_rope(
                      code, qp, kp, vp, kcp, vcp, cp, sp, pp, smp, bp, clp, op, (int)b, (int)hq,
                      (int)hkv, (int)d, (int)mb, bs, nb, rows, qs, ks, scale, st);
                }),
                out);
}

// Element strides of [B, S, H, D] between sequences and between positions (a
// dimension of one element gets its contiguous stride), or false where the
// prefill kernel cannot read the tensor in place (the rule of ops._head_rows).
bool head_rows(const at::Tensor &t, int64_t *seq, int64_t *row) {
  const int64_t b = t.size(0), s = t.size(1), h = t.size(2), d = t.size(3);
  *row = s > 1 ? t.stride(1) : h * d;
  *seq = b > 1 ? t.stride(0) : *row * s;
  if (t.is_contiguous()) return true;
  return t.stride(3) == 1 && (h == 1 || t.stride(2) == d) && *row >= h * d && *row % 8 == 0 &&
         *seq >= 0 && *seq % 8 == 0 && *row < (1 << 30) && *row * (s + 512) < (1 << 30) &&
         (uintptr_t)t.data_ptr() % 16 == 0;
}

PyObject *prefill_attention(PyObject *const *a) {
  const at::Tensor *q = plain(a[0]), *k = plain(a[1]), *v = plain(a[2]);
  float scale;
  if (!q || !k || !v || !as_float(a[3], &scale) || q->dim() != 4 || k->dim() != 4) return declined();
  const int code = dtype_code(*q);
  const int64_t b = q->size(0), s = q->size(1), hq = q->size(2), d = q->size(3), hkv = k->size(2);
  if (code < 0 || k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type() ||
      k->device() != q->device() || v->device() != q->device() || v->sizes() != k->sizes() ||
      k->size(0) != b || k->size(1) != s || k->size(3) != d || !fits_int({b, s, hq, hkv, d}))
    return declined();
  int64_t qs, qr, ks, kr, vs, vr;
  if (!head_rows(*q, &qs, &qr) || !head_rows(*k, &ks, &kr) || !head_rows(*v, &vs, &vr) || ks != vs ||
      kr != vr)
    return declined();
  const c10::DeviceGuard guard(q->device());
  at::Tensor out = at::empty({b, s, hq, d}, q->options());
  const void *qp = q->data_ptr(), *kp = k->data_ptr(), *vp = v->data_ptr();
  void *op = out.data_ptr(), *st = stream_of(q->device());
  return result(launch([&] {
                  return g_lib.mce_prefill_attention_strided(code, qp, kp, vp, op, (int)b, (int)s,
                                                             (int)hq, (int)hkv, (int)d, qs, qr, ks,
                                                             kr, scale, st);
                }),
                out);
}

PyObject *prefill_attention_paged(PyObject *const *a) {
  const at::Tensor *q = plain(a[0]), *kc = plain(a[1]), *vc = plain(a[2]), *bt = plain(a[3]),
                   *cl = plain(a[4]);
  float scale;
  if (!q || !bt || !as_float(a[5], &scale) || !PyBool_Check(a[6]) || q->dim() != 4 ||
      !q->is_contiguous() || bt->dim() != 2)
    return declined();
  const int code = dtype_code(*q);
  const int64_t b = q->size(0), s = q->size(1), hq = q->size(2), d = q->size(3), w = bt->size(1);
  if (code < 0 || b < 1 || s < 1 || !pools(kc, vc, *q, -1, d) || !ints(bt, b * w, q->device()) ||
      !ints(cl, b, q->device()) || !fits_int({b, s, hq, d, w, kc->size(1), kc->size(2)}))
    return declined();
  const int hkv = (int)kc->size(2), bs = (int)kc->size(1);
  const c10::DeviceGuard guard(q->device());
  at::Tensor out = at::empty_like(*q);
  const size_t ws_bytes = a[6] == Py_True ? g_lib.mce_prefill_attention_paged_workspace_size(
                                                (int)b, (int)s, (int)hq, hkv)
                                          : 0;
  const Workspace ws(ws_bytes, *q);
  const void *qp = q->data_ptr(), *kp = kc->data_ptr(), *vp = vc->data_ptr();
  const int32_t *bp = (const int32_t *)bt->data_ptr(), *cp = (const int32_t *)cl->data_ptr();
  void *op = out.data_ptr(), *st = stream_of(q->device());
  const int64_t nb = kc->size(0);
  return result(launch([&] {
                  return g_lib.mce_prefill_attention_paged(code, qp, kp, vp, bp, cp, op, (int)b, (int)s,
                                                           (int)hq, hkv, (int)d, (int)w, bs, nb, scale,
                                                           ws.ptr, ws_bytes, st);
                }),
                out);
}

// x, norm weight (None: plain projection), eps, weight, out (None: a new
// tensor), epilogue code
PyObject *projection(PyObject *const *a) {
  const at::Tensor *x = plain(a[0]), *nw = a[1] == Py_None ? nullptr : plain(a[1]),
                   *w = plain(a[3]), *o = a[4] == Py_None ? nullptr : plain(a[4]);
  int64_t epi;
  float eps = 0.f;
  if (!x || !w || (a[1] != Py_None && (!nw || !as_float(a[2], &eps))) || (a[4] != Py_None && !o) ||
      !as_int(a[5], &epi) || x->dim() != 2 || w->dim() != 2)
    return declined();
  const int code = dtype_code(*x);
  const int64_t m = x->size(0), k = x->size(1);
  if (code < 0 || w->scalar_type() != x->scalar_type() || w->device() != x->device() ||
      w->size(1) != k || x->stride(1) != 1 || !w->is_contiguous() ||
      (epi == MCE_EPI_SWIGLU && w->size(0) % 2 != 0) || (epi == MCE_EPI_ADD && !o))
    return declined();
  const int64_t n = epi == MCE_EPI_SWIGLU ? w->size(0) / 2 : w->size(0);
  if (!fits_int({m, n, k})) return declined();
  if (nw && (nw->scalar_type() != x->scalar_type() || nw->device() != x->device() || nw->dim() != 1 ||
             nw->numel() != k || !nw->is_contiguous()))
    return declined();
  if (o && (o->scalar_type() != x->scalar_type() || o->device() != x->device() || o->dim() != 2 ||
            o->size(0) != m || o->size(1) != n || o->stride(1) != 1))
    return declined();
  const c10::DeviceGuard guard(x->device());
  at::Tensor out = o ? *o : at::empty({m, n}, x->options());
  const void *xp = x->data_ptr(), *np = nw ? nw->data_ptr() : nullptr, *wp = w->data_ptr();
  void *op = out.data_ptr(), *st = stream_of(x->device());
  const int64_t xs = x->stride(0), os = out.stride(0);
  const int rc = launch([&] {
    return nw ? g_lib.mce_rmsnorm_decode_gemm(code, xp, np, eps, wp, op, (int)m, (int)n, (int)k, xs, os,
                                              (int)epi, st)
              : g_lib.mce_decode_gemm(code, xp, wp, op, (int)m, (int)n, (int)k, xs, os, (int)epi, st);
  });
  if (rc != MCE_OK || !o) return result(rc, out);
  Py_INCREF(a[4]);
  return a[4];
}

// x, weight, out (None: a new tensor), epilogue code, norm weight (None), eps:
// the projection of a prompt; returns out, or the normalised rows with a norm.
// Declined where autograd or a dispatch mode has to see the library GEMM.
PyObject *prompt_gemm(PyObject *const *a) {
  const at::Tensor *x = plain(a[0]), *w = plain(a[1]), *o = a[2] == Py_None ? nullptr : plain(a[2]),
                   *nw = a[4] == Py_None ? nullptr : plain(a[4]);
  int64_t epi;
  float eps = 0.f;
  if (!x || !w || (a[2] != Py_None && !o) || (a[4] != Py_None && (!nw || !as_float(a[5], &eps))) ||
      !as_int(a[3], &epi) || x->dim() != 2 || w->dim() != 2 ||
      c10::impl::TorchDispatchModeTLS::any_modes_set())
    return declined();
  if (at::GradMode::is_enabled())
    for (const at::Tensor *t : {x, w, o, nw})
      if (t && t->requires_grad()) return declined();
  const int code = dtype_code(*x);
  const int64_t m = x->size(0), k = x->size(1);
  if (code < 0 || w->scalar_type() != x->scalar_type() || w->device() != x->device() ||
      w->size(1) != k || x->stride(1) != 1 || !w->is_contiguous() ||
      (epi == MCE_EPI_SWIGLU && w->size(0) % 2 != 0) || (epi == MCE_EPI_ADD && !o))
    return declined();
  const int64_t n = epi == MCE_EPI_SWIGLU ? w->size(0) / 2 : w->size(0);
  if (!fits_int({m, n, k})) return declined();
  if (o && (o->scalar_type() != x->scalar_type() || o->device() != x->device() || o->dim() != 2 ||
            o->size(0) != m || o->size(1) != n || o->stride(1) != 1))
    return declined();
  if (nw && (nw->scalar_type() != x->scalar_type() || nw->device() != x->device() || nw->dim() != 1 ||
             nw->numel() != n || !nw->is_contiguous()))
    return declined();
  if (!g_lib.mce_prompt_gemm_takes((int)m, (int)n, (int)k, (int)epi)) return declined();
  const c10::DeviceGuard guard(x->device());
  at::Tensor out = o ? *o : at::empty({m, n}, x->options());
  at::Tensor normed;
  if (nw) normed = at::empty({m, n}, x->options());
  const size_t ws_bytes = g_lib.mce_prompt_gemm_workspace_size((int)m, (int)n, (int)k, (int)epi);
  const Workspace ws(ws_bytes, *x);
  const void *xp = x->data_ptr(), *wp = w->data_ptr(), *np = nw ? nw->data_ptr() : nullptr;
  void *op = out.data_ptr(), *yp = nw ? normed.data_ptr() : nullptr, *st = stream_of(x->device());
  const int64_t xs = x->stride(0), os = out.stride(0);
  const int rc = launch([&] {
    return g_lib.mce_prompt_gemm(code, xp, wp, op, (int)m, (int)n, (int)k, xs, os, (int)epi, np, eps, yp,
                                 ws.ptr, ws_bytes, st);
  });
  return result(rc, nw ? normed : out);
}

// C++ exceptions (torch's allocator, a bad device) become Python errors.
template <PyObject *(*OP)(PyObject *const *), int N>
PyObject *call(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != N) {
    PyErr_Format(PyExc_TypeError, "%d arguments expected, got %zd", N, n);
    return nullptr;
  }
  if (!g_bound) return declined();
  try {
    return OP(args);
  } catch (const c10::OutOfMemoryError &) {
    return declined();  // ops.py repeats the allocation and reports it as torch does
  } catch (const std::exception &e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

// bind({name: address}): every entry point of MCE_NATIVE_ENTRIES
PyObject *bind(PyObject *, PyObject *dict) {
  if (!PyDict_Check(dict)) {
    PyErr_SetString(PyExc_TypeError, "bind takes a dict of entry point addresses");
    return nullptr;
  }
  Entries e;
  PyObject *v;
#define X(name)                                                         \
  v = PyDict_GetItemString(dict, #name);                                \
  if (!v) {                                                             \
    PyErr_SetString(PyExc_KeyError, #name);                             \
    return nullptr;                                                     \
  }                                                                     \
  e.name = (decltype(e.name))PyLong_AsVoidPtr(v);                       \
  if (!e.name) {                                                        \
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, #name);    \
    return nullptr;                                                     \
  }
  MCE_NATIVE_ENTRIES(X)
#undef X
  g_lib = e;
  g_bound = true;
  Py_RETURN_NONE;
}

PyObject *entries(PyObject *, PyObject *) {
  PyObject *l = PyList_New(0);
  if (!l) return nullptr;
#define X(name)                                        \
  {                                                    \
    PyObject *s = PyUnicode_FromString(#name);         \
    if (!s || PyList_Append(l, s) != 0) return nullptr; \
    Py_DECREF(s);                                      \
  }
  MCE_NATIVE_ENTRIES(X)
#undef X
  return l;
}

#define OP(name, fn, n) \
  {name, (PyCFunction)(void (*)(void))(_PyCFunctionFast)call<fn, n>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"bind", bind, METH_O, nullptr},
    {"entries", entries, METH_NOARGS, nullptr},
    OP("rmsnorm", rmsnorm, 3),
    OP("swiglu", swiglu, 1),
    OP("paged_kv_store", paged_kv_store, 5),
    OP("paged_attention_decode", paged_attention_decode, 8),
    OP("rope_inplace", rope_inplace, 5),
    OP("rope_kv_store", rope_kv_store, 10),
    OP("decode_rope_attention", decode_rope_attention, 13),
    OP("prefill_attention", prefill_attention, 4),
    OP("prefill_attention_paged", prefill_attention_paged, 7),
    OP("projection", projection, 6),
    OP("prompt_gemm", prompt_gemm, 6),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods,
                      nullptr,               nullptr,   nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }
