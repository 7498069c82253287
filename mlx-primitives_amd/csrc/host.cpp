// Native host path of the Python layer: one call per operator that checks the
// tensors' layout, allocates outputs and workspace through torch's caching
// allocator and enqueues the C-ABI call on the caller's stream. What it covers
// is the ordinary case (plain tensors on one device, aligned layouts); anything
// else returns None and the Python layer takes its general path, so a call
// accepts, refuses and returns the same either way.
//
// Why: the same steps in Python (strides, data pointers, some thirty ctypes
// arguments) took as long as a small kernel: a flash_attention forward 15 us of
// host time, a decode step of append, rotation and attention 64 us, forward and
// backward 75 us (an idle box; busy ones up to twice that).
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>

#include "mpx_attn.h"
#include "mpx_attn_sched.h"

namespace {

// Entries of the loaded library, by address (init).
#define MPX_ENTRIES(X)                                                                      \
  X(mpx_attn_fwd_lse)                                                                       \
  X(mpx_attn_fwd_dropout)                                                                   \
  X(mpx_attn_fwd_workspace_bytes)                                                           \
  X(mpx_attn_bwd)                                                                           \
  X(mpx_attn_bwd_dropout)                                                                   \
  X(mpx_attn_bwd_grouped)                                                                   \
  X(mpx_attn_bwd_workspace_bytes)                                                           \
  X(mpx_attn_bwd_grouped_workspace_bytes)                                                   \
  X(mpx_attn_bwd_ds_preferred)                                                              \
  X(mpx_paged_decode_gqa)                                                                   \
  X(mpx_paged_decode_workspace_bytes)                                                       \
  X(mpx_paged_prefill_gqa)                                                                  \
  X(mpx_paged_prefill_workspace_bytes)                                                      \
  X(mpx_kv_append)                                                                          \
  X(mpx_kv_append_rope)                                                                     \
  X(mpx_rope_at)
struct Api {
#define X(name) decltype(&::name) name = nullptr;
  MPX_ENTRIES(X)
#undef X
} api;

// A plain torch tensor on a device (no subclass, no functorch or dispatch
// wrapper, storage present), or nullptr.
const at::Tensor* plain(PyObject* obj) {
  if (!THPVariable_CheckExact(obj) && Py_TYPE(obj) != (PyTypeObject*)ParameterClass) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(obj);
  static const c10::DispatchKeySet wrapped({c10::DispatchKey::Python,
                                            c10::DispatchKey::FuncTorchGradWrapper,
                                            c10::DispatchKey::FuncTorchBatched,
                                            c10::DispatchKey::Functionalize});
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage() ||
      t.key_set().has_any(wrapped))
    return nullptr;
  return &t;
}

int dtype_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return MPX_F32;
    case at::kHalf: return MPX_F16;
    case at::kBFloat16: return MPX_BF16;
    default: return -1;
  }
}

// The kernels' layout: last dimension contiguous, other strides multiples of
// 16 bytes, 16-byte aligned.
bool aligned_rows(const at::Tensor& t, int vec) {
  const int64_t n = t.dim();
  if (t.stride(n - 1) != 1 || ((uintptr_t)t.data_ptr() & 15u) != 0) return false;
  for (int64_t i = 0; i + 1 < n; ++i)
    if (t.stride(i) % vec != 0) return false;
  return true;
}

bool int32_contiguous(const at::Tensor& t) {
  return t.scalar_type() == at::kInt && t.is_contiguous();
}

struct Strides {
  int64_t s[3];
  // (batch, head, seq) of a 4-D tensor in BSHD or BHSD order
  Strides(const at::Tensor& t, bool bshd)
      : s{t.stride(0), t.stride(bshd ? 2 : 1), t.stride(bshd ? 1 : 2)} {}
};

at::Tensor bytes(size_t n, const at::Tensor& like) {
  return at::empty({(int64_t)(n < 16 ? 16 : n)}, like.options().dtype(at::kByte));
}

// f() without the GIL, which is taken back also when f throws (data_ptr() of
// some tensors does).
template <class F>
int call(F&& f) {
  struct Released {
    PyThreadState* const state = PyEval_SaveThread();
    ~Released() { PyEval_RestoreThread(state); }
  } released;
  return f();
}

// An argument as the general path's int(...) and ctypes read it: what has
// __int__, __index__ or __trunc__ (masks and windows come as the user gave
// them: floats, numpy scalars), of which the low bits count.
int64_t as_int(PyObject* o) {
  if (PyLong_Check(o)) return (int64_t)PyLong_AsUnsignedLongLongMask(o);
  PyObject* const x = PyNumber_Long(o);
  if (!x) return -1;
  const int64_t v = (int64_t)PyLong_AsUnsignedLongLongMask(x);
  Py_DECREF(x);
  return v;
}
double as_float(PyObject* o) { return PyFloat_AsDouble(o); }

bool wrong_count(Py_ssize_t n, Py_ssize_t want) {
  if (n == want) return false;
  PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
  return true;
}

// attn_fwd(q, k, v, bshd, D, scale, causal, wl, wr, want_lse, drop_p, seed, stream)
//   -> o, (o, lse), an error code, or None
PyObject* attn_fwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (wrong_count(n, 13)) return nullptr;
  const at::Tensor *q = plain(a[0]), *k = plain(a[1]), *v = plain(a[2]);
  if (!q || !k || !v || q->device() != k->device() || q->device() != v->device()) Py_RETURN_NONE;
  const int code = dtype_code(*q);
  const bool bshd = as_int(a[3]) != 0;
  const int D = (int)as_int(a[4]);
  const int vec = code == MPX_F32 ? 4 : 8;
  for (const at::Tensor* t : {q, k, v})
    if (t->dim() != 4 || t->size(3) != D || dtype_code(*t) != code || code < 0 ||
        !aligned_rows(*t, vec))
      Py_RETURN_NONE;
  const double scale = as_float(a[5]), drop_p = as_float(a[10]);
  const int causal = (int)as_int(a[6]), wl = (int)as_int(a[7]), wr = (int)as_int(a[8]);
  const bool want_lse = as_int(a[9]) != 0;
  const uint64_t seed = PyLong_AsUnsignedLongLongMask(a[11]);
  void* stream = PyLong_AsVoidPtr(a[12]);
  if (PyErr_Occurred()) return nullptr;
  const int hd = bshd ? 2 : 1, sd = bshd ? 1 : 2;
  const int B = (int)q->size(0), H = (int)q->size(hd), Sq = (int)q->size(sd);
  const int H_kv = (int)k->size(hd), Sk = (int)k->size(sd);
  at::Tensor o = at::empty(q->sizes(), q->options()), lse, ws;
  if (want_lse) lse = at::empty({B, H, Sq}, q->options().dtype(at::kFloat));
  const size_t need = api.mpx_attn_fwd_workspace_bytes(B, H, Sq, Sk, D, causal, wl, wr, code);
  if (need) ws = bytes(need, *q);
  const Strides qs(*q, bshd), ks(*k, bshd), vs(*v, bshd), os(o, bshd);
  float* const lp = want_lse ? lse.data_ptr<float>() : nullptr;
  void* const wp = need ? ws.data_ptr() : nullptr;
  const int rc = call([&] {
    if (drop_p >= 0)
      return api.mpx_attn_fwd_dropout(q->data_ptr(), k->data_ptr(), v->data_ptr(), o.data_ptr(), lp,
                                      qs.s, ks.s, vs.s, os.s, B, H, H_kv, Sq, Sk, D, (float)scale,
                                      causal, wl, wr, code, (float)drop_p, seed, wp, need, stream);
    return api.mpx_attn_fwd_lse(q->data_ptr(), k->data_ptr(), v->data_ptr(), o.data_ptr(), lp,
                                qs.s, ks.s, vs.s, os.s, B, H, H_kv, Sq, Sk, D, (float)scale,
                                causal, wl, wr, code, wp, need, stream);
  });
  if (rc != MPX_OK) return PyLong_FromLong(rc);
  if (!want_lse) return THPVariable_Wrap(std::move(o));
  PyObject* out = PyTuple_New(2);
  if (!out) return nullptr;
  PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(o)));
  PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(lse)));
  return out;
  END_HANDLE_TH_ERRORS
}

// attn_bwd(q, k, v, o, dout, lse, bshd, scale, causal, wl, wr, drop_p, seed,
//   may_store_ds, stream) -> (dq, dk, dv), an error code, or None (also where
// the stored-dS schedule is the better one, or memory for parts is short)
PyObject* attn_bwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (wrong_count(n, 15)) return nullptr;
  const at::Tensor* t[6];
  for (int i = 0; i < 6; ++i) {
    t[i] = plain(a[i]);
    if (!t[i] || t[i]->device() != t[0]->device()) Py_RETURN_NONE;
  }
  const at::Tensor &q = *t[0], &k = *t[1], &v = *t[2], &o = *t[3], &dout = *t[4], &lse = *t[5];
  const int code = dtype_code(q);
  if (code < 0 || q.dim() != 4) Py_RETURN_NONE;
  const int vec = code == MPX_F32 ? 4 : 8, D = (int)q.size(3);
  for (int i = 0; i < 5; ++i)
    if (t[i]->dim() != 4 || t[i]->size(3) != D || dtype_code(*t[i]) != code ||
        !aligned_rows(*t[i], vec))
      Py_RETURN_NONE;
  if (lse.scalar_type() != at::kFloat || !lse.is_contiguous() || dout.sizes() != q.sizes() ||
      o.sizes() != q.sizes())
    Py_RETURN_NONE;
  const bool bshd = as_int(a[6]) != 0;
  const double scale = as_float(a[7]), drop_p = as_float(a[11]);
  const int causal = (int)as_int(a[8]), wl = (int)as_int(a[9]), wr = (int)as_int(a[10]);
  const uint64_t seed = PyLong_AsUnsignedLongLongMask(a[12]);
  const bool may_store = as_int(a[13]) != 0;
  void* stream = PyLong_AsVoidPtr(a[14]);
  if (PyErr_Occurred()) return nullptr;
  const int hd = bshd ? 2 : 1, sd = bshd ? 1 : 2;
  const int B = (int)q.size(0), H = (int)q.size(hd), Sq = (int)q.size(sd);
  const int H_kv = (int)k.size(hd), Sk = (int)k.size(sd);
  if (may_store && drop_p >= 0 &&
      api.mpx_attn_bwd_ds_preferred(B, H, H_kv, Sq, Sk, D, code, wl))
    Py_RETURN_NONE;
  const bool grouped = H != H_kv;
  const size_t need =
      grouped ? api.mpx_attn_bwd_grouped_workspace_bytes(B, H, H_kv, Sq, Sk, D, code, wl)
              : api.mpx_attn_bwd_workspace_bytes(B, H, Sq);
  at::Tensor ws;
  try {
    ws = bytes(need, q);
  } catch (const c10::OutOfMemoryError&) {
    Py_RETURN_NONE;
  }
  at::Tensor dq = at::empty(q.sizes(), q.options()), dk = at::empty(k.sizes(), k.options()),
             dv = at::empty(v.sizes(), v.options());
  const Strides s[8] = {{q, bshd}, {k, bshd}, {v, bshd}, {o, bshd},
                        {dout, bshd}, {dq, bshd}, {dk, bshd}, {dv, bshd}};
  const float* const lp = lse.data_ptr<float>();
  const int rc = call([&] {
#define MPX_BWD_ARGS                                                                          \
  q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), dout.data_ptr(), lp, dq.data_ptr(), \
      dk.data_ptr(), dv.data_ptr(), s[0].s, s[1].s, s[2].s, s[3].s, s[4].s, s[5].s, s[6].s,   \
      s[7].s, B, H, H_kv, Sq, Sk, D, (float)scale, causal, wl, wr, code
    if (grouped)
      return api.mpx_attn_bwd_grouped(MPX_BWD_ARGS, drop_p >= 0 ? (float)drop_p : 0.f, seed,
                                      ws.data_ptr(), need, stream);
    if (drop_p >= 0)
      return api.mpx_attn_bwd_dropout(MPX_BWD_ARGS, (float)drop_p, seed, ws.data_ptr(), need,
                                      stream);
    return api.mpx_attn_bwd(MPX_BWD_ARGS, ws.data_ptr(), need, stream);
#undef MPX_BWD_ARGS
  });
  if (rc != MPX_OK) return PyLong_FromLong(rc);
  PyObject* out = PyTuple_New(3);
  if (!out) return nullptr;
  PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(dq)));
  PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(dk)));
  PyTuple_SET_ITEM(out, 2, THPVariable_Wrap(std::move(dv)));
  return out;
  END_HANDLE_TH_ERRORS
}

// paged_attend(q, k_pool, v_pool, tables, lens, slopes or None, scale, causal,
//   stream) -> o, an error code, or None; the caller has checked the shapes.
// Decode for one query per sequence, else prefill (head dims of the kernels).
PyObject* paged_attend(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (wrong_count(n, 9)) return nullptr;
  const at::Tensor* t[6];
  for (int i = 0; i < 6; ++i) {
    t[i] = nullptr;
    if (i == 5 && a[5] == Py_None) break;
    t[i] = plain(a[i]);
    if (!t[i] || t[i]->device() != t[0]->device()) Py_RETURN_NONE;
  }
  const at::Tensor &q = *t[0], &kp = *t[1], &vp = *t[2], &bt = *t[3], &cl = *t[4];
  const int code = dtype_code(q);
  const int vec = code == MPX_F32 ? 4 : 8;
  if (code < 0 || q.dim() != 4 || kp.dim() != 4 || q.size(3) % vec != 0 || !aligned_rows(q, vec) ||
      !kp.is_contiguous() || !vp.is_contiguous() || !int32_contiguous(bt) ||
      !int32_contiguous(cl) ||
      (t[5] && (t[5]->scalar_type() != at::kFloat || !t[5]->is_contiguous())))
    Py_RETURN_NONE;
  const double scale = as_float(a[6]);
  const int B = (int)q.size(0), Sq = (int)q.size(1), H = (int)q.size(2), D = (int)q.size(3);
  const int causal = Sq == 1 ? 0 : (int)as_int(a[7]);  // (decode takes no mask)
  void* stream = PyLong_AsVoidPtr(a[8]);
  if (PyErr_Occurred()) return nullptr;
  const int nb = (int)kp.size(0), bs = (int)kp.size(1), H_kv = (int)kp.size(2);
  const int mb = (int)bt.size(1);
  at::Tensor o = at::empty(q.sizes(), q.options());
  const size_t need =
      Sq == 1 ? api.mpx_paged_decode_workspace_bytes(B, H, D, bs, mb)
              : api.mpx_paged_prefill_workspace_bytes(B, Sq, H, D, bs, mb, causal, code);
  at::Tensor ws = bytes(need, q);
  const int64_t qs[3] = {q.stride(0), q.stride(2), q.stride(1)};
  const int64_t os[3] = {o.stride(0), o.stride(2), o.stride(1)};
  const float* const sl = t[5] ? t[5]->data_ptr<float>() : nullptr;
  const int rc = call([&] {
    if (Sq != 1)
      return api.mpx_paged_prefill_gqa(q.data_ptr(), kp.data_ptr(), vp.data_ptr(),
                                       bt.data_ptr<int32_t>(), cl.data_ptr<int32_t>(), sl,
                                       o.data_ptr(), qs, os, B, Sq, H, H_kv, D, nb, bs, mb,
                                       (float)scale, causal, code, ws.data_ptr(),
                                       (size_t)ws.numel(), stream);
    return api.mpx_paged_decode_gqa(q.data_ptr(), kp.data_ptr(), vp.data_ptr(),
                                    bt.data_ptr<int32_t>(), cl.data_ptr<int32_t>(), sl,
                                    o.data_ptr(), qs, os, B, H, H_kv, D, nb, bs, mb, (float)scale,
                                    code, ws.data_ptr(), (size_t)ws.numel(), stream);
  });
  if (rc != MPX_OK) return PyLong_FromLong(rc);
  return THPVariable_Wrap(std::move(o));
  END_HANDLE_TH_ERRORS
}

// kv_append(k, v, k_pool, v_pool, tables, starts, counts, errors, cos or None,
//   sin or None, stream) -> an error code, or None; clears errors first; the
// caller has checked the shapes
PyObject* kv_append(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (wrong_count(n, 11)) return nullptr;
  const bool rope = a[8] != Py_None;
  const at::Tensor* t[10];
  for (int i = 0; i < (rope ? 10 : 8); ++i) {
    t[i] = plain(a[i]);
    if (!t[i] || t[i]->device() != t[0]->device()) Py_RETURN_NONE;
  }
  const at::Tensor &k = *t[0], &v = *t[1], &kp = *t[2], &vp = *t[3], &bt = *t[4];
  const int code = dtype_code(kp);
  const int vec = code == MPX_F32 ? 4 : 8;
  if (code < 0 || k.dim() != 4 || v.dim() != 4 || !aligned_rows(k, vec) || !aligned_rows(v, vec) ||
      !int32_contiguous(bt) || !int32_contiguous(*t[5]) || !int32_contiguous(*t[6]) ||
      !int32_contiguous(*t[7]))
    Py_RETURN_NONE;
  if (rope && (!t[8]->is_contiguous() || !t[9]->is_contiguous() || dtype_code(*t[8]) < 0))
    Py_RETURN_NONE;
  void* stream = PyLong_AsVoidPtr(a[10]);
  if (PyErr_Occurred()) return nullptr;
  t[7]->zero_();
  const int B = (int)k.size(0), T = (int)k.size(1), H = (int)k.size(2), D = (int)k.size(3);
  const int nb = (int)kp.size(0), bs = (int)kp.size(1), mb = (int)bt.size(1);
  const int64_t ks[3] = {k.stride(0), k.stride(1), k.stride(2)};
  const int64_t vs[3] = {v.stride(0), v.stride(1), v.stride(2)};
  const int rc = call([&] {
    if (rope)
      return api.mpx_kv_append_rope(
          k.data_ptr(), v.data_ptr(), kp.data_ptr(), vp.data_ptr(), bt.data_ptr<int32_t>(),
          t[5]->data_ptr<int32_t>(), t[6]->data_ptr<int32_t>(), ks, vs, B, T, H, D, nb, bs, mb,
          code, t[8]->data_ptr(), t[9]->data_ptr(), (int)t[8]->size(0), dtype_code(*t[8]),
          t[7]->data_ptr<int32_t>(), stream);
    return api.mpx_kv_append(k.data_ptr(), v.data_ptr(), kp.data_ptr(), vp.data_ptr(),
                             bt.data_ptr<int32_t>(), t[5]->data_ptr<int32_t>(),
                             t[6]->data_ptr<int32_t>(), ks, vs, B, T, H, D, nb, bs, mb, code,
                             t[7]->data_ptr<int32_t>(), stream);
  });
  return PyLong_FromLong(rc);
  END_HANDLE_TH_ERRORS
}

// rope_at(x, cos, sin, positions, errors, stream) -> out, an error code, or
// None; clears errors first; the caller has checked the shapes
PyObject* rope_at(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (wrong_count(n, 6)) return nullptr;
  const at::Tensor* t[5];
  for (int i = 0; i < 5; ++i) {
    t[i] = plain(a[i]);
    if (!t[i] || t[i]->device() != t[0]->device()) Py_RETURN_NONE;
  }
  const at::Tensor& x = *t[0];
  const int code = dtype_code(x), cdt = dtype_code(*t[1]);
  if (code < 0 || cdt < 0 || x.dim() != 4 || !aligned_rows(x, code == MPX_F32 ? 4 : 8) ||
      !t[1]->is_contiguous() || !t[2]->is_contiguous() || !int32_contiguous(*t[3]) ||
      !int32_contiguous(*t[4]))
    Py_RETURN_NONE;
  void* stream = PyLong_AsVoidPtr(a[5]);
  if (PyErr_Occurred()) return nullptr;
  at::Tensor out = at::empty(x.sizes(), x.options());
  t[4]->zero_();
  const int64_t xs[3] = {x.stride(0), x.stride(1), x.stride(2)};
  const int64_t os[3] = {out.stride(0), out.stride(1), out.stride(2)};
  const int rc = call([&] {
    return api.mpx_rope_at(x.data_ptr(), out.data_ptr(), t[1]->data_ptr(), t[2]->data_ptr(), xs, os,
                           (int)x.size(0), (int)x.size(1), (int)x.size(2), (int)x.size(3),
                           t[3]->data_ptr<int32_t>(), (int)t[1]->size(0), code, cdt,
                           t[4]->data_ptr<int32_t>(), stream);
  });
  if (rc != MPX_OK) return PyLong_FromLong(rc);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// init({entry name: address}): the library that the calls go to.
PyObject* init(PyObject*, PyObject* dict) {
#define X(name)                                                                       \
  {                                                                                   \
    PyObject* p = PyDict_GetItemString(dict, #name);                                  \
    if (!p) {                                                                         \
      PyErr_SetString(PyExc_KeyError, #name);                                         \
      return nullptr;                                                                 \
    }                                                                                 \
    api.name = reinterpret_cast<decltype(&::name)>(PyLong_AsVoidPtr(p));              \
    if (PyErr_Occurred()) return nullptr;                                             \
  }
  MPX_ENTRIES(X)
#undef X
  Py_RETURN_NONE;
}

// entries(): the names that init needs.
PyObject* entries(PyObject*, PyObject*) {
  PyObject* out = PyList_New(0);
  if (!out) return nullptr;
#define X(name)                                             \
  {                                                         \
    PyObject* s = PyUnicode_FromString(#name);              \
    if (!s || PyList_Append(out, s) != 0) {                 \
      Py_XDECREF(s);                                        \
      Py_DECREF(out);                                       \
      return nullptr;                                       \
    }                                                       \
    Py_DECREF(s);                                           \
  }
  MPX_ENTRIES(X)
#undef X
  return out;
}

#define FAST(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST(attn_fwd),  FAST(attn_bwd), FAST(paged_attend),
                         FAST(kv_append), FAST(rope_at),  {"init", init, METH_O, nullptr},
                         {"entries", entries, METH_NOARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_mpx_host", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__mpx_host() { return PyModule_Create(&module); }
