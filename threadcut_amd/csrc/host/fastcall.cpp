// The call paths of a decode step in native code: what the Python wrappers do
// per call (tensor checks, stride arrays, workspace, the library call) for the
// calls that need no special treatment, without ctypes.
//
// Each function returns None (or False) for anything else: another device
// than the current one, a tensor subclass, a shape, type or stride that the
// kernels refuse. The Python wrapper then takes the call, checks it in full
// and raises what there is to raise. Nothing is enqueued in that case: the
// library validates before it launches.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/GradMode.h>
#include <c10/core/InferenceMode.h>
#include <c10/core/impl/DeviceGuardImplInterface.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../../include/threadcut_hip.h"

namespace {

constexpr int64_t kHeadDim = 128;

bool dtype_code(const at::Tensor& t, int* code) {
  if (t.scalar_type() == at::kHalf) { *code = TC_DTYPE_F16; return true; }
  if (t.scalar_type() == at::kBFloat16) { *code = TC_DTYPE_BF16; return true; }
  return false;
}

// A plain torch.Tensor with memory on the current GPU. The device is looked
// up once per call and passed on.
const at::Tensor* tensor(PyObject* o, const c10::Device& dev) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.has_storage() || t.device() != dev || t.layout() != at::kStrided) return nullptr;
  return &t;
}

bool current(PyObject* o, c10::Device* dev) {
  if (!THPVariable_CheckExact(o)) return false;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda()) return false;
  const c10::impl::DeviceGuardImplInterface* impl = c10::impl::getDeviceGuardImpl(c10::DeviceType::CUDA);
  *dev = t.device();
  return impl->getDevice() == *dev;
}

int64_t stride(const at::Tensor& t, int i) { return t.size(i) > 1 ? t.stride(i) : 0; }

// The cache's [B, Hkv, N, 128] strides; a single token's row keeps its own length.
void cache_strides(const at::Tensor& t, int64_t st[3]) {
  st[0] = stride(t, 0);
  st[1] = stride(t, 1);
  st[2] = t.size(2) > 1 ? t.stride(2) : kHeadDim;
}

bool same_type(const at::Tensor& q, const at::Tensor& t) { return t.scalar_type() == q.scalar_type(); }

// q [B, Hq, 1, 128] of a decode step with its KV heads: batch, heads, group
// and the strides of its [B, Hkv, G, 128] view.
struct Query {
  int64_t b, hq, hkv, g;
  int64_t st[3];
  int dt;
};

bool query(const at::Tensor& q, const at::Tensor& k, Query* x) {
  if (q.dim() != 4 || k.dim() != 4 || q.size(2) != 1 || q.size(3) != kHeadDim || k.size(3) != kHeadDim) return false;
  if (!dtype_code(q, &x->dt) || !same_type(q, k) || q.stride(3) != 1 || k.stride(3) != 1) return false;
  x->b = q.size(0);
  x->hq = q.size(1);
  x->hkv = k.size(1);
  if (x->b < 1 || k.size(0) != x->b || x->hkv < 1 || x->hq % x->hkv) return false;
  x->g = x->hq / x->hkv;
  if (x->g < 1 || x->g > 8) return false;
  const int64_t sh = q.stride(1);
  x->st[0] = stride(q, 0);
  x->st[1] = x->hkv > 1 ? x->g * sh : 0;
  x->st[2] = x->g > 1 ? sh : 0;
  return true;
}

// The split plan's workspace; false for a plan that the library refuses.
bool workspace(const at::Tensor& q, const Query& x, int64_t n, int64_t split, int ragged, at::Tensor* ws) {
  const int s = tc_decode_num_splits(static_cast<int>(x.b), static_cast<int>(x.hkv), n, static_cast<int>(split), ragged);
  if (s < 0) return false;
  const size_t bytes = tc_decode_workspace_bytes(static_cast<int>(x.b), static_cast<int>(x.hkv), static_cast<int>(x.g),
                                                 static_cast<int>(kHeadDim), s);
  *ws = at::empty({static_cast<int64_t>(bytes < 16 ? 16 : bytes)}, q.options().dtype(at::kByte).requires_grad(false));
  return true;
}

// The output [B, 1, Hq, 128] and its strides as [B, Hkv, G, 128].
at::Tensor output(const at::Tensor& q, const Query& x, int64_t st[3]) {
  st[0] = x.hq * kHeadDim;
  st[1] = x.g * kHeadDim;
  st[2] = kHeadDim;
  return at::empty({x.b, 1, x.hq, kHeadDim}, q.options().requires_grad(false));
}

void* raw_stream(PyObject* o) { return reinterpret_cast<void*>(static_cast<uintptr_t>(PyLong_AsUnsignedLongLong(o))); }

// A new token's rows [B, Hkv, 128] or [B, Hkv, 1, 128] and their (batch, head) strides.
bool new_rows(const at::Tensor& t, const at::Tensor& q, const Query& x, int64_t st[2]) {
  if (!same_type(q, t) || (t.dim() != 3 && !(t.dim() == 4 && t.size(2) == 1))) return false;
  if (t.size(0) != x.b || t.size(1) != x.hkv || t.size(-1) != kHeadDim || t.stride(-1) != 1) return false;
  st[0] = stride(t, 0);
  st[1] = stride(t, 1);
  return true;
}

// decode(query [b, hq, 1, d], key, value [b, hkv, n, d], scale, stream) -> out [b, 1, hq, d] or None
PyObject* decode(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  c10::Device dev(c10::DeviceType::CPU);
  if (n_args != 5 || !current(a[0], &dev)) Py_RETURN_NONE;
  const at::Tensor *q = tensor(a[0], dev), *k = tensor(a[1], dev), *v = tensor(a[2], dev);
  Query x;
  if (!q || !k || !v || !query(*q, *k, &x)) Py_RETURN_NONE;
  if (!same_type(*q, *v) || v->sizes() != k->sizes() || v->stride(3) != 1) Py_RETURN_NONE;
  const double scale = PyFloat_AsDouble(a[3]);
  void* stream = raw_stream(a[4]);
  if (PyErr_Occurred()) return nullptr;
  int64_t so[3], sk[3], sv[3];
  cache_strides(*k, sk);
  cache_strides(*v, sv);
  const int64_t n = k->size(2);
  at::Tensor ws;
  if (!workspace(*q, x, n, 0, 0, &ws)) Py_RETURN_NONE;
  at::Tensor out = output(*q, x, so);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = tc_decode_attention(q->const_data_ptr(), x.st, k->const_data_ptr(), sk, v->const_data_ptr(), sv, nullptr, n,
                           static_cast<int>(x.b), static_cast<int>(x.hkv), static_cast<int>(x.g), kHeadDim, x.dt,
                           static_cast<float>(scale), 0, ws.mutable_data_ptr(), ws.numel(), out.mutable_data_ptr(), so,
                           stream);
  Py_END_ALLOW_THREADS
  if (rc != TC_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// decode_append(query, k_buf, v_buf [b, hkv, cap, d], k_new, v_new, n or pos, scale, stream) -> out or None.
// A whole number: the rows go to token n - 1; an int32 [b] tensor: to token pos[b] (the plan is the capacity's).
PyObject* decode_append(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  c10::Device dev(c10::DeviceType::CPU);
  if (n_args != 8 || !current(a[0], &dev)) Py_RETURN_NONE;
  const at::Tensor *q = tensor(a[0], dev), *k = tensor(a[1], dev), *v = tensor(a[2], dev), *kn = tensor(a[3], dev),
                   *vn = tensor(a[4], dev);
  Query x;
  int64_t so[3], sk[3], sv[3], skn[2], svn[2];
  if (!q || !k || !v || !kn || !vn || !query(*q, *k, &x)) Py_RETURN_NONE;
  if (!same_type(*q, *v) || v->sizes() != k->sizes() || v->stride(3) != 1) Py_RETURN_NONE;
  if (!new_rows(*kn, *q, x, skn) || !new_rows(*vn, *q, x, svn)) Py_RETURN_NONE;
  const int64_t cap = k->size(2);
  const int32_t* pos = nullptr;
  int64_t n = cap;
  if (THPVariable_Check(a[5])) {
    const at::Tensor* p = tensor(a[5], dev);
    if (!p || p->scalar_type() != at::kInt || p->dim() != 1 || p->size(0) != x.b || !p->is_contiguous()) Py_RETURN_NONE;
    pos = static_cast<const int32_t*>(p->const_data_ptr());
  } else {
    n = PyLong_AsLongLong(a[5]);
  }
  const double scale = PyFloat_AsDouble(a[6]);
  void* stream = raw_stream(a[7]);
  if (PyErr_Occurred()) return nullptr;
  if (n < 1 || n > cap) Py_RETURN_NONE;
  cache_strides(*k, sk);
  cache_strides(*v, sv);
  at::Tensor ws;
  if (!workspace(*q, x, n, 0, 0, &ws)) Py_RETURN_NONE;
  at::Tensor out = output(*q, x, so);
  const int b = static_cast<int>(x.b), hkv = static_cast<int>(x.hkv), g = static_cast<int>(x.g);
  const float sc = static_cast<float>(scale);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = pos ? tc_decode_append_attention_at(q->const_data_ptr(), x.st, k->mutable_data_ptr(), sk, v->mutable_data_ptr(),
                                           sv, kn->const_data_ptr(), skn, vn->const_data_ptr(), svn, pos, cap, b, hkv,
                                           g, kHeadDim, x.dt, sc, 0, ws.mutable_data_ptr(), ws.numel(),
                                           out.mutable_data_ptr(), so, stream)
           : tc_decode_append_attention(q->const_data_ptr(), x.st, k->mutable_data_ptr(), sk, v->mutable_data_ptr(), sv,
                                        kn->const_data_ptr(), skn, vn->const_data_ptr(), svn, n, b, hkv, g, kHeadDim,
                                        x.dt, sc, 0, ws.mutable_data_ptr(), ws.numel(), out.mutable_data_ptr(), so,
                                        stream);
  Py_END_ALLOW_THREADS
  if (rc != TC_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// paged_append(q [b, hkv, g, d], k_pool, v_pool [pages, hkv, P, d], table [b, tiles, 4], counts [b], k_new, v_new,
// out or None, scale, stream) -> out [b, hkv, g, d] or None: PagedKV.decode_append's call.
PyObject* paged_append(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  c10::Device dev(c10::DeviceType::CPU);
  if (n_args != 10 || !current(a[0], &dev)) Py_RETURN_NONE;
  const at::Tensor* t[7];
  for (int i = 0; i < 7; ++i)
    if (!(t[i] = tensor(a[i], dev))) Py_RETURN_NONE;
  const at::Tensor &q = *t[0], &kp = *t[1], &vp = *t[2], &tab = *t[3], &cnt = *t[4], &kn = *t[5], &vn = *t[6];
  Query x;
  if (q.dim() != 4 || kp.dim() != 4 || q.size(3) != kHeadDim || kp.size(3) != kHeadDim || !dtype_code(q, &x.dt)) Py_RETURN_NONE;
  if (!same_type(q, kp) || !same_type(q, vp) || vp.sizes() != kp.sizes() || vp.strides() != kp.strides()) Py_RETURN_NONE;
  x.b = q.size(0);
  x.hkv = q.size(1);
  x.g = q.size(2);
  if (x.b < 1 || kp.size(1) != x.hkv || q.stride(3) != 1 || kp.stride(3) != 1 || tab.dim() != 3 || tab.size(0) != x.b) Py_RETURN_NONE;
  int64_t skn[2], svn[2];
  if (!new_rows(kn, q, x, skn) || !new_rows(vn, q, x, svn)) Py_RETURN_NONE;
  const double scale = PyFloat_AsDouble(a[8]);
  void* stream = raw_stream(a[9]);
  if (PyErr_Occurred()) return nullptr;
  at::Tensor out;
  if (a[7] == Py_None) {
    out = at::empty_like(q);
  } else {
    const at::Tensor* o = tensor(a[7], dev);
    if (!o || o->sizes() != q.sizes() || !same_type(q, *o) || o->stride(3) != 1) Py_RETURN_NONE;
    out = *o;
  }
  const int64_t tiles = tab.size(1);
  at::Tensor ws;
  if (!workspace(q, x, 16 * tiles, 0, x.b > 1, &ws)) Py_RETURN_NONE;
  const int64_t sq[3] = {q.stride(0), q.stride(1), q.stride(2)}, sp[3] = {kp.stride(0), kp.stride(1), kp.stride(2)},
                so[3] = {out.stride(0), out.stride(1), out.stride(2)};
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = tc_decode_paged_append_attention(
      q.const_data_ptr(), sq, kp.mutable_data_ptr(), vp.mutable_data_ptr(), sp, static_cast<int>(kp.size(0)),
      static_cast<int>(kp.size(2)), static_cast<const int32_t*>(tab.const_data_ptr()),
      static_cast<const int32_t*>(cnt.const_data_ptr()), tiles, kn.const_data_ptr(), skn, vn.const_data_ptr(), svn,
      static_cast<int>(x.b), static_cast<int>(x.hkv), static_cast<int>(x.g), kHeadDim, x.dt, static_cast<float>(scale), 0,
      ws.mutable_data_ptr(), ws.numel(), out.mutable_data_ptr(), so, stream);
  Py_END_ALLOW_THREADS
  if (rc != TC_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// True for a tensor whose in-place copy torch would record or refuse: autograd (a view of a tracked buffer counts),
// a forward-mode tangent, an inference tensor outside inference mode.
bool recorded(const at::Tensor& t) {
  return (c10::GradMode::is_enabled() && t.requires_grad()) || t._fw_grad(0).defined() ||
         (t.is_inference() && !c10::InferenceMode::is_enabled());
}

// True while something sees every operation of this thread: torch.jit.trace, a dispatch mode and a functorch transform
// each include a dispatch key of their own.
bool watched() {
  return !(c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set).empty();
}

// append_rows(k_buf, v_buf [b, h, cap, d], row0, k, v [b, h, rows, d], stream) -> bool: new tokens' rows into both
// buffers. Autograd is told of the write (the buffers' versions), as torch's copy would tell it.
PyObject* append_rows(PyObject*, PyObject* const* a, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  c10::Device dev(c10::DeviceType::CPU);
  if (n_args != 6 || !current(a[0], &dev)) Py_RETURN_FALSE;
  const at::Tensor *kb = tensor(a[0], dev), *vb = tensor(a[1], dev), *k = tensor(a[3], dev), *v = tensor(a[4], dev);
  int dt;
  if (!kb || !vb || !k || !v || kb->dim() != 4 || k->dim() != 4 || !dtype_code(*kb, &dt)) Py_RETURN_FALSE;
  if (vb->sizes() != kb->sizes() || vb->strides() != kb->strides() || v->sizes() != k->sizes()) Py_RETURN_FALSE;
  for (const at::Tensor* t : {k, v})
    if (!same_type(*kb, *t) || t->size(0) != kb->size(0) || t->size(1) != kb->size(1) || t->size(3) != kHeadDim ||
        kb->size(3) != kHeadDim || t->stride(3) != 1)
      Py_RETURN_FALSE;
  // Writes that autograd, tracing, a dispatch mode or a functorch transform would record stay torch's copies.
  for (const at::Tensor* t : {kb, vb, k, v})
    if (recorded(*t)) Py_RETURN_FALSE;
  if (watched()) Py_RETURN_FALSE;
  const int64_t row0 = PyLong_AsLongLong(a[2]);
  void* stream = raw_stream(a[5]);
  if (PyErr_Occurred()) return nullptr;
  const int64_t sk[3] = {k->stride(0), k->stride(1), k->stride(2)}, sv[3] = {v->stride(0), v->stride(1), v->stride(2)},
                sb[3] = {kb->stride(0), kb->stride(1), kb->stride(2)};
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = tc_append_rows(k->const_data_ptr(), sk, v->const_data_ptr(), sv, kb->mutable_data_ptr(), vb->mutable_data_ptr(),
                      sb, kb->size(2), row0, static_cast<int>(kb->size(0)), static_cast<int>(kb->size(1)), k->size(2),
                      kHeadDim, dt, stream);
  Py_END_ALLOW_THREADS
  if (rc != TC_OK) Py_RETURN_FALSE;
  if (!kb->is_inference()) kb->unsafeGetTensorImpl()->bump_version();
  if (!vb->is_inference()) vb->unsafeGetTensorImpl()->bump_version();
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

PyCFunction fast(PyObject* (*f)(PyObject*, PyObject* const*, Py_ssize_t)) {
  return reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(f));
}

}  // namespace

PyMODINIT_FUNC PyInit__fast() {
  static PyMethodDef methods[] = {
      {"decode", fast(decode), METH_FASTCALL, "decode(query, key, value, scale, stream) -> out or None"},
      {"decode_append", fast(decode_append), METH_FASTCALL,
       "decode_append(query, k_buf, v_buf, k_new, v_new, n_or_pos, scale, stream) -> out or None"},
      {"paged_append", fast(paged_append), METH_FASTCALL,
       "paged_append(q, k_pool, v_pool, table, counts, k_new, v_new, out, scale, stream) -> out or None"},
      {"append_rows", fast(append_rows), METH_FASTCALL, "append_rows(k_buf, v_buf, row0, k, v, stream) -> bool"},
      {nullptr, nullptr, 0, nullptr}};
  static PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fast", "Native call paths of the wrappers.", -1, methods};
  PyObject* m = PyModule_Create(&module);
  // The torch whose headers these paths were compiled with: they read its tensors in place, so they serve no other.
  if (m && PyModule_AddStringConstant(m, "torch_version", TC_TORCH_VERSION) < 0) Py_CLEAR(m);
  return m;
}
