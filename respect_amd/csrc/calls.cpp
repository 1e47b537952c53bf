// The kernel wrappers' common case in native code: a CPython module that checks a
// call's tensors, allocates its outputs, finds the current stream and makes the
// one C-ABI call (include/respect_amd.h) -- what the Python wrappers do with
// ctypes, whose argument conversions and per-tensor checks cost 10 to 20
// microseconds on calls whose kernels take 3.
//
// Every function returns None for a call it does not take (another type, dtype,
// device, layout or shape rule): the Python wrapper then goes through its own
// checks, which copy what needs a copy and raise what has to be raised.  A nonzero
// status of the C ABI comes back as an int.  Nothing is kept between calls.
#include <Python.h>

#include <cmath>
#include <vector>

#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include "respect_amd.h"

namespace {

using at::Tensor;

// o as a plain CUDA tensor of dtype `t` with readable storage, else null.
const Tensor* plain(PyObject* o, at::ScalarType t = at::kBFloat16) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor& x = THPVariable_Unpack(o);
  if (!x.defined() || !x.is_cuda() || x.scalar_type() != t || x.layout() != at::kStrided || !x.has_storage()) return nullptr;
  return &x;
}

// The layout as_kernel_input passes through: 16-byte aligned, contiguous last
// dimension, the other strides multiples of 8 elements.
bool aligned(const Tensor& t) {
  if (reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16) return false;
  const int64_t n = t.dim();
  if (n && t.stride(n - 1) != 1 && t.size(n - 1) != 1) return false;
  for (int64_t i = 0; i + 1 < n; ++i)
    if (t.stride(i) % 8) return false;
  return true;
}

const Tensor* input(PyObject* o) {
  const Tensor* t = plain(o);
  return t && aligned(*t) ? t : nullptr;
}

const void* ptr(const Tensor& t) { return t.const_data_ptr(); }

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

Tensor empty_like_of(const Tensor& x, at::IntArrayRef shape, at::ScalarType t = at::kBFloat16) {
  return at::empty(shape, x.options().dtype(t).requires_grad(false));
}

// Rows [M, N] of a tensor whose leading dimensions merge into one without a copy.
bool rows_of(const Tensor& t, int64_t& m, int64_t& n, int64_t& stride) {
  const int64_t d = t.dim();
  if (d < 1) return false;
  n = t.size(d - 1);
  if (n == 0) return false;   // the wrapper refuses rows of no elements
  if (d == 2) {
    m = t.size(0);
    stride = t.stride(0);
    return t.stride(1) == 1;
  }
  if (!t.is_contiguous()) return false;
  m = t.numel() / n;
  stride = n;
  return true;
}

bool fits_int(int64_t v) { return v >= 0 && v <= 0x7fffffff; }

// The C-ABI call without the GIL.  f also asks torch for pointers and the stream, which
// may throw (a tensor without readable memory): the destructor takes the GIL back first.
struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  NoGil() = default;
  NoGil(const NoGil&) = delete;
  ~NoGil() { PyEval_RestoreThread(state); }
};

template <class F>
int call(F&& f) {
  NoGil no_gil;
  return f();
}

PyObject* wrap(Tensor&& t) { return THPVariable_Wrap(std::move(t)); }

bool number(PyObject* o, double& v) {
  if (!PyFloat_CheckExact(o) && !PyLong_CheckExact(o)) return false;
  v = PyFloat_AsDouble(o);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

#define NOT_TAKEN Py_RETURN_NONE
#define STATUS(rc) \
  if ((rc) != RSPX_OK) return PyLong_FromLong(rc)

// silu_mul(g, u)
PyObject* silu_mul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2) NOT_TAKEN;
  const Tensor *g = input(a[0]), *u = input(a[1]);
  if (!g || !u || g->sizes() != u->sizes() || g->device() != u->device()) NOT_TAKEN;
  int64_t m, f, sg, mu, fu, su;
  if (!rows_of(*g, m, f, sg) || !rows_of(*u, mu, fu, su) || !fits_int(m) || !fits_int(f)) NOT_TAKEN;
  Tensor y = empty_like_of(*g, g->sizes());
  const int rc = call([&] { return rspx_silu_mul(ptr(*g), sg, ptr(*u), su, y.data_ptr(), f, (int)m, (int)f, stream_of(*g)); });
  STATUS(rc);
  return wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// rmsnorm(x, w, eps)
PyObject* rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  double eps;
  if (n != 3 || !number(a[2], eps)) NOT_TAKEN;
  const Tensor *x = input(a[0]), *w = input(a[1]);
  int64_t m, k, sx;
  if (!x || !w || x->device() != w->device() || w->dim() != 1 || !rows_of(*x, m, k, sx) || w->size(0) != k || k % 8 ||
      !fits_int(m) || !fits_int(k))
    NOT_TAKEN;
  Tensor y = empty_like_of(*x, x->sizes());
  const int rc =
      call([&] { return rspx_rmsnorm(ptr(*x), sx, ptr(*w), y.data_ptr(), k, (int)m, (int)k, (float)eps, stream_of(*x)); });
  STATUS(rc);
  return wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// q [T, HQ, D], k [T, HK, D], wq / wk [D], cos / sin [T, D] as the kernels take them.
struct QK {
  const Tensor *q, *k, *wq, *wk, *cos, *sin;
  int64_t T, HQ, HK, D;
  bool read(PyObject* const* a) {   // q, k, wq, wk
    q = input(a[0]);
    k = input(a[1]);
    wq = input(a[2]);
    wk = input(a[3]);
    if (!q || !k || !wq || !wk || q->dim() != 3 || k->dim() != 3 || wq->dim() != 1 || wk->dim() != 1) return false;
    T = q->size(0);
    HQ = q->size(1);
    D = q->size(2);
    HK = k->size(1);
    return k->size(0) == T && k->size(2) == D && wq->size(0) == D && wk->size(0) == D && D % 16 == 0 && fits_int(T) &&
           fits_int(HQ) && fits_int(HK) && q->device() == k->device() && q->device() == wq->device() &&
           q->device() == wk->device();
  }
  bool tables(PyObject* c, PyObject* s) {
    cos = input(c);
    sin = input(s);
    return cos && sin && cos->dim() == 2 && cos->size(0) == T && cos->size(1) == D && sin->sizes() == cos->sizes() &&
           cos->stride(0) == sin->stride(0) && cos->device() == q->device() && sin->device() == q->device();
  }
};

// qk_norm_rope(q, k, wq, wk, eps, cos, sin)
PyObject* qk_norm_rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  double eps;
  QK s;
  if (n != 7 || !number(a[4], eps) || !s.read(a) || !s.tables(a[5], a[6])) NOT_TAKEN;
  Tensor qo = empty_like_of(*s.q, {s.T, s.HQ, s.D}), ko = empty_like_of(*s.q, {s.T, s.HK, s.D});
  const int rc = call([&] {
    return rspx_qk_norm_rope(ptr(*s.q), s.q->stride(0), s.q->stride(1), ptr(*s.k), s.k->stride(0), s.k->stride(1),
                             ptr(*s.wq), ptr(*s.wk), ptr(*s.cos), ptr(*s.sin), s.cos->stride(0), qo.data_ptr(),
                             ko.data_ptr(), (int)s.T, (int)s.HQ, (int)s.HK, (int)s.D, (float)eps, stream_of(*s.q));
  });
  STATUS(rc);
  return Py_BuildValue("(NN)", wrap(std::move(qo)), wrap(std::move(ko)));
  END_HANDLE_TH_ERRORS
}

// rmsnorm_qk_norm_rope(x, w, eps, q, k, wq, wk, qk_eps, cos, sin)
PyObject* rmsnorm_qk_norm_rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  double eps, qeps;
  QK s;
  if (n != 10 || !number(a[2], eps) || !number(a[7], qeps)) NOT_TAKEN;
  const Tensor *x = input(a[0]), *w = input(a[1]);
  int64_t m, k, sx;
  if (!x || !w || x->device() != w->device() || w->dim() != 1 || !rows_of(*x, m, k, sx) || w->size(0) != k || k % 8 ||
      k > 16384 || !fits_int(m))
    NOT_TAKEN;
  if (!s.read(a + 3) || !s.tables(a[8], a[9]) || s.q->device() != x->device()) NOT_TAKEN;
  Tensor y = empty_like_of(*x, x->sizes());
  Tensor qo = empty_like_of(*s.q, {s.T, s.HQ, s.D}), ko = empty_like_of(*s.q, {s.T, s.HK, s.D});
  const int rc = call([&] {
    return rspx_rmsnorm_qk_norm_rope(ptr(*x), sx, ptr(*w), y.data_ptr(), k, (int)m, (int)k, (float)eps, ptr(*s.q),
                                     s.q->stride(0), s.q->stride(1), ptr(*s.k), s.k->stride(0), s.k->stride(1),
                                     ptr(*s.wq), ptr(*s.wk), ptr(*s.cos), ptr(*s.sin), s.cos->stride(0), qo.data_ptr(),
                                     ko.data_ptr(), (int)s.T, (int)s.HQ, (int)s.HK, (int)s.D, (float)qeps,
                                     stream_of(*x));
  });
  STATUS(rc);
  return Py_BuildValue("(NNN)", wrap(std::move(y)), wrap(std::move(qo)), wrap(std::move(ko)));
  END_HANDLE_TH_ERRORS
}

// rope(x, cos, sin)
PyObject* rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3) NOT_TAKEN;
  const Tensor *x = input(a[0]), *c = input(a[1]), *s = input(a[2]);
  if (!x || !c || !s || x->dim() != 4 || c->dim() != 3 || !c->is_contiguous() || !s->is_contiguous() ||
      s->sizes() != c->sizes() || c->device() != x->device() || s->device() != x->device())
    NOT_TAKEN;
  const int64_t B = x->size(0), H = x->size(1), L = x->size(2), D = x->size(3);
  if (c->size(0) != B || c->size(1) != L || c->size(2) != D || !fits_int(B) || !fits_int(H) || !fits_int(L) || !fits_int(D))
    NOT_TAKEN;
  Tensor y = empty_like_of(*x, x->sizes());
  const int rc = call([&] {
    return rspx_rope(ptr(*x), x->stride(0), x->stride(1), x->stride(2), ptr(*c), ptr(*s), c->stride(0), c->stride(1),
                     y.data_ptr(), (int)B, (int)H, (int)L, (int)D, stream_of(*x));
  });
  STATUS(rc);
  return wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// add_sq(r, h)
PyObject* add_sq(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2) NOT_TAKEN;
  const Tensor *r = input(a[0]), *h = input(a[1]);
  if (!r || !h || r->dim() != 2 || r->sizes() != h->sizes() || !r->is_contiguous() || !h->is_contiguous() ||
      r->device() != h->device() || !fits_int(r->size(0)) || !fits_int(r->size(1)) || r->size(1) == 0)
    NOT_TAKEN;
  const int64_t m = r->size(0), k = r->size(1);
  Tensor x = empty_like_of(*r, {m, k}), sq = empty_like_of(*r, {m, k}, at::kFloat);
  const int rc = call([&] {
    return rspx_add_sq(ptr(*r), r->stride(0), ptr(*h), h->stride(0), x.data_ptr(), x.stride(0), sq.data_ptr<float>(),
                       sq.stride(0), (int)m, (int)k, stream_of(*r));
  });
  STATUS(rc);
  return Py_BuildValue("(NN)", wrap(std::move(x)), wrap(std::move(sq)));
  END_HANDLE_TH_ERRORS
}

// norm_apply(xs, var, w, eps): norm_from after its mean.
PyObject* norm_apply(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  double eps;
  if (n != 4 || !number(a[3], eps)) NOT_TAKEN;
  const Tensor *x = input(a[0]), *w = input(a[2]), *v = plain(a[1], at::kFloat);
  if (!x || !w || !v || x->dim() != 2 || v->dim() != 1 || w->dim() != 1 || !x->is_contiguous() || !v->is_contiguous() ||
      !w->is_contiguous() || v->size(0) != x->size(0) || w->size(0) != x->size(1) || x->device() != w->device() ||
      x->device() != v->device() || !fits_int(x->size(0)) || !fits_int(x->size(1)))
    NOT_TAKEN;
  const int64_t m = x->size(0), k = x->size(1);
  Tensor y = empty_like_of(*x, {m, k});
  const int rc = call([&] {
    return rspx_norm_apply(ptr(*x), x->stride(0), v->const_data_ptr<float>(), ptr(*w), y.data_ptr(), y.stride(0), (int)m,
                           (int)k, (float)eps, stream_of(*x));
  });
  STATUS(rc);
  return wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// rope_vision(x, cos, sin) with fp32 tables [L, D]
PyObject* rope_vision(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3) NOT_TAKEN;
  const Tensor *x = input(a[0]), *c = plain(a[1], at::kFloat), *s = plain(a[2], at::kFloat);
  if (!x || !c || !s || x->dim() != 3 || c->dim() != 2 || !c->is_contiguous() || !s->is_contiguous() ||
      c->sizes() != s->sizes() || c->size(0) != x->size(0) || c->size(1) != x->size(2) || c->device() != x->device() ||
      s->device() != x->device())
    NOT_TAKEN;
  const int64_t L = x->size(0), NH = x->size(1), D = x->size(2);
  if (!fits_int(L) || !fits_int(NH) || !fits_int(D)) NOT_TAKEN;
  Tensor y = empty_like_of(*x, {L, NH, D});
  const int rc = call([&] {
    return rspx_rope_vision(ptr(*x), x->stride(0), x->stride(1), c->const_data_ptr<float>(), s->const_data_ptr<float>(),
                            c->stride(0), y.data_ptr(), (int)L, (int)NH, (int)D, stream_of(*x));
  });
  STATUS(rc);
  return wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// The scratch tensor of (device, current stream, tag) in the workspace dict of
// respect_amd._lib if it holds at least `need` bytes (else the Python side makes
// it).  A reference is held over the call: another thread may replace the entry.
bool scratch(PyObject* dict, const Tensor& x, PyObject* tag, int64_t need, Tensor& out) {
  if (!PyDict_CheckExact(dict)) return false;
  PyObject* key = Py_BuildValue("(iKO)", (int)x.device().index(), (unsigned long long)stream_of(x), tag);
  PyObject* ws = key ? PyDict_GetItemWithError(dict, key) : nullptr;   // borrowed
  Py_XDECREF(key);
  if (!ws || !THPVariable_CheckExact(ws)) {
    PyErr_Clear();
    return false;
  }
  out = THPVariable_Unpack(ws);
  return out.numel() >= need;
}

// linear(x, w, N, K, tiled, fp32, workspaces, tag): w a tensor, or the buffer of
// a tiled weight (tiled = True).
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8) NOT_TAKEN;
  const Tensor *x = input(a[0]), *w = input(a[1]);
  const bool tiled = a[4] == Py_True, fp32 = a[5] == Py_True;
  if (!x || !w || x->device() != w->device()) NOT_TAKEN;
  int64_t m, k, sx, N, K;
  if (!rows_of(*x, m, k, sx) || !fits_int(m)) NOT_TAKEN;
  if (tiled) {
    N = PyLong_AsLongLong(a[2]);
    K = PyLong_AsLongLong(a[3]);
  } else {
    if (w->dim() != 2) NOT_TAKEN;
    N = w->size(0);
    K = w->size(1);
  }
  if (K != k || !fits_int(N) || !fits_int(K) || N == 0 || K == 0) NOT_TAKEN;
  const int64_t need = rspx_linear_workspace_bytes((int)m, (int)N, (int)K);
  if (need < 0) NOT_TAKEN;
  Tensor ws;
  if (need > 0 && !scratch(a[6], *x, a[7], need, ws)) NOT_TAKEN;
  std::vector<int64_t> shape(x->sizes().begin(), x->sizes().end());
  shape.back() = N;
  Tensor y = empty_like_of(*x, shape, fp32 ? at::kFloat : at::kBFloat16);
  const int rc = call([&] {
    return rspx_linear(ptr(*x), sx, ptr(*w), tiled ? RSPX_TILED : w->stride(0), y.data_ptr(), N, (int)m, (int)N, (int)K,
                       fp32 ? 1 : 0, need > 0 ? ws.data_ptr() : nullptr, need > 0 ? ws.numel() : 0, stream_of(*x));
  });
  STATUS(rc);
  return wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// trie_attn(q, kp, vp, kn, vn, msk, sm_scale, workspaces, tag): a new [H, M, D]
// result, automatic work split.
PyObject* trie_attn(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 9) NOT_TAKEN;
  const Tensor* t[5];
  for (int i = 0; i < 5; ++i) {
    t[i] = input(a[i]);
    if (!t[i] || t[i]->dim() != 3 || t[i]->device() != t[0]->device()) NOT_TAKEN;
  }
  const Tensor *q = t[0], *kp = t[1], *vp = t[2], *kn = t[3], *vn = t[4];
  const Tensor* msk = plain(a[5], at::kBool);
  if (!msk) msk = plain(a[5], at::kByte);
  if (!msk || msk->dim() != 2 || msk->device() != q->device()) NOT_TAKEN;
  const int64_t H = q->size(0), M = q->size(1), D = q->size(2), HK = kp->size(0), P = kp->size(1), NN = kn->size(1);
  if (kp->size(2) != D || vp->sizes() != kp->sizes() || kn->size(0) != HK || kn->size(2) != D ||
      vn->sizes() != kn->sizes() || msk->size(0) != M || msk->size(1) != NN)
    NOT_TAKEN;
  for (int64_t v : {H, M, D, HK, P, NN})
    if (!fits_int(v)) NOT_TAKEN;
  double scale;
  if (a[6] == Py_None) scale = std::pow((double)D, -0.5);
  else if (!number(a[6], scale)) NOT_TAKEN;
  const int64_t need = rspx_trie_attn_workspace_bytes((int)H, (int)HK, (int)M, (int)P, (int)D);
  if (need < 0) NOT_TAKEN;
  Tensor ws;
  if (!scratch(a[7], *q, a[8], need, ws)) NOT_TAKEN;
  Tensor y = empty_like_of(*q, {H, M, D});
  const int rc = call([&] {
    return rspx_trie_attn(ptr(*q), q->stride(0), q->stride(1), ptr(*kp), kp->stride(0), kp->stride(1), ptr(*vp),
                          vp->stride(0), vp->stride(1), ptr(*kn), kn->stride(0), kn->stride(1), ptr(*vn), vn->stride(0),
                          vn->stride(1), static_cast<const uint8_t*>(ptr(*msk)), msk->stride(0), msk->stride(1),
                          y.data_ptr(), y.stride(0), y.stride(1), (int)H, (int)HK, (int)M, (int)P, (int)NN, (int)D,
                          (float)scale, ws.data_ptr(), ws.numel(), 0, stream_of(*q));
  });
  STATUS(rc);
  return wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

#define FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST(silu_mul), FAST(rmsnorm), FAST(qk_norm_rope), FAST(rmsnorm_qk_norm_rope),
                         FAST(rope),     FAST(add_sq),  FAST(norm_apply),   FAST(rope_vision),
                         FAST(linear),   FAST(trie_attn), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// VERSION and TORCH: what the module was compiled against, for respect_amd._lib to compare.
PyMODINIT_FUNC PyInit__calls() {
  PyObject* m = PyModule_Create(&module);
  if (m && (PyModule_AddStringConstant(m, "VERSION", RSPX_VERSION) || PyModule_AddStringConstant(m, "TORCH", TORCH_VERSION))) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
