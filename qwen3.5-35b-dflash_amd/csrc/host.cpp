// Native form of the plain calls of ops.py: argument checks, output and scratch allocation and the C entry in one
// Python call.
//
// A decoded token's projection is 3.5 us of device time and was 17 us of Python (validation, descriptors, ctypes, two
// allocations); a 16-token GDN layer 89 us of device time behind 156 us of it.  Every function here takes the arguments
// of its namesake in ops.py, does what that does when they are plain (exact torch.Tensor and bank types, contiguous, on
// one ROCm device, no dispatch or function mode active) and returns None otherwise, before anything is launched; ops.py
// then takes its own path, which decides and reports as it always did.  A call that its entry refuses raises what ops.py
// would (_lib.check).  No state but the entry points' addresses, the two bank types and that function, set once by
// bind().  The GIL is released while an entry enqueues.
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <c10/core/GradMode.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/dflash_hip.h"

namespace {

PyTypeObject* g_packed_type = nullptr;
PyTypeObject* g_shared_type = nullptr;
PyObject* g_check = nullptr;

struct Entries {
  decltype(&dflash_qlinear_workspace_bytes) qlinear_workspace_bytes;
  decltype(&dflash_qlinear_w4a16) qlinear;
  decltype(&dflash_qlinear_w4a16_f32) qlinear_f32;
  decltype(&dflash_moe_workspace_bytes) moe_workspace_bytes;
  decltype(&dflash_moe_w4a16) moe;
  decltype(&dflash_moe_w4a16_residual) moe_residual;
  decltype(&dflash_gdn_workspace_bytes) gdn_workspace_bytes;
  decltype(&dflash_gdn_mixer) gdn;
  decltype(&dflash_gdn_commit) commit;
  decltype(&dflash_rms_norm) rms_norm;
  decltype(&dflash_attention_workspace_bytes) attention_workspace_bytes;
  decltype(&dflash_attention_mixer) attention;
} g_entry;

// _lib.check of a nonzero status: raises DflashError with the library's message
PyObject* refused(const char* entry, int status) {
  PyObject* r = PyObject_CallFunction(g_check, "si", entry, status);
  if (r) PyErr_SetString(PyExc_SystemError, "a refused call was not reported");
  Py_XDECREF(r);
  return nullptr;
}

bool plain_state() { return !c10::impl::dispatch_mode_enabled() && !at::impl::torch_function_mode_enabled(); }

// A plain dense device tensor, or null.
const at::Tensor* tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided ||
      !(t.unsafeGetTensorImpl()->key_set() & at::kTensorSubclassLike).empty())
    return nullptr;
  return &t;
}

// ops._tracked: a gradient is asked for, or a forward-mode tangent is carried
bool tracked(const at::Tensor& t) {
  return (t.requires_grad() && c10::GradMode::is_enabled()) || t.unsafeGetTensorImpl()->_fw_grad(0, t).defined();
}

// What ops._as accepts: this dtype, shape and device, contiguous, 16-byte aligned.
const at::Tensor* exactly(PyObject* o, at::ScalarType dtype, at::IntArrayRef shape, at::Device device) {
  const at::Tensor* t = tensor(o);
  if (!t || t->scalar_type() != dtype || t->sizes() != shape || t->device() != device || !t->is_contiguous() ||
      reinterpret_cast<uintptr_t>(t->data_ptr()) % 16)
    return nullptr;
  return t;
}

// The descriptor of a valid bank of `ndim` dimensions on `device` (PackedW4.validate and ops._desc).
bool bank(PyObject* o, int64_t ndim, at::Device device, dflash_w4* d) {
  if (Py_TYPE(o) != g_packed_type) return false;
  const at::Tensor* p = tensor(PyTuple_GET_ITEM(o, 0));
  const at::Tensor* s = tensor(PyTuple_GET_ITEM(o, 1));
  PyObject* group = PyTuple_GET_ITEM(o, 2);
  PyObject* layout = PyTuple_GET_ITEM(o, 3);
  if (!p || !s || !PyLong_CheckExact(group) || !PyUnicode_Check(layout)) return false;
  const long g = PyLong_AsLong(group);
  if (g != 128 && g != 256) {
    PyErr_Clear();
    return false;
  }
  const bool tiled = PyUnicode_CompareWithASCIIString(layout, "tiled") == 0;
  if (!tiled && PyUnicode_CompareWithASCIIString(layout, "portable") != 0) return false;
  if (p->scalar_type() != at::kByte || p->dim() != ndim || s->dim() != ndim || p->device() != device ||
      s->device() != device || !p->is_contiguous() || !s->is_contiguous())
    return false;
  if (s->scalar_type() != at::kBFloat16 && s->scalar_type() != at::kFloat) return false;
  const int64_t n = p->size(-2), k = p->size(-1) * 2;
  if (k % g || s->size(-1) != k / g || s->size(-2) != n || (ndim == 3 && s->size(0) != p->size(0))) return false;
  if (tiled && (n % 16 || k % 128)) return false;
  *d = dflash_w4{};
  d->packed = p->data_ptr();
  d->scales = s->data_ptr();
  d->experts = ndim == 3 ? p->size(0) : 1;
  d->rows = n;
  d->cols = k;
  d->group_size = g;
  d->scale_dtype = s->scalar_type() == at::kFloat ? DFLASH_DTYPE_F32 : DFLASH_DTYPE_BF16;
  d->layout = tiled ? DFLASH_LAYOUT_TILED : DFLASH_LAYOUT_PORTABLE;
  return true;
}

at::Tensor make(at::IntArrayRef shape, at::ScalarType dtype, at::Device device) {
  return at::empty(shape, at::TensorOptions().dtype(dtype).device(device));
}
at::Tensor bytes(size_t n, at::Device device) {
  return make({static_cast<int64_t>(std::max<size_t>(n, 256))}, at::kByte, device);
}
void* stream_of(at::Device device) { return c10::hip::getCurrentHIPStream(device.index()).stream(); }

// The caller's workspace, or a new one; false: a workspace that ops._workspace refuses.
bool workspace_of(PyObject* o, size_t need, at::Device device, at::Tensor* ws) {
  if (o == Py_None) {
    *ws = bytes(need, device);
    return true;
  }
  const at::Tensor* t = tensor(o);
  if (!t || t->scalar_type() != at::kByte || t->device() != device || static_cast<size_t>(t->numel()) < need) return false;
  *ws = *t;
  return true;
}

bool want(Py_ssize_t got, Py_ssize_t n) {
  if (got == n) return true;
  PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", n, got);
  return false;
}

// linear(x, weight, f32_out)
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!want(n, 3)) return nullptr;
  const at::Tensor* x = plain_state() ? tensor(a[0]) : nullptr;
  dflash_w4 w;
  if (!x || x->scalar_type() != at::kBFloat16 || x->dim() < 1 || !x->is_contiguous() || x->numel() == 0 ||
      !bank(a[1], 2, x->device(), &w) || x->size(-1) != w.cols)
    Py_RETURN_NONE;
  const bool f32 = a[2] == Py_True;
  const int64_t m = x->numel() / w.cols;
  std::vector<int64_t> shape = x->sizes().vec();
  shape.back() = w.rows;
  at::Tensor y = make(shape, f32 ? at::kFloat : at::kBFloat16, x->device());
  const at::Tensor ws = bytes(g_entry.qlinear_workspace_bytes(m, w.cols, w.group_size), x->device());
  void* st = stream_of(x->device());
  int status;
  Py_BEGIN_ALLOW_THREADS
  if (f32) status = g_entry.qlinear_f32(x->data_ptr(), m, &w, static_cast<float*>(y.data_ptr()), ws.data_ptr(), ws.numel(), st);
  else status = g_entry.qlinear(x->data_ptr(), m, &w, y.data_ptr(), ws.data_ptr(), ws.numel(), st);
  Py_END_ALLOW_THREADS
  if (status) return refused(f32 ? "dflash_qlinear_w4a16_f32" : "dflash_qlinear_w4a16", status);
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// moe(hidden, gate_up, down, top_k, router_weight, shared, workspace, residual): residual None: the bf16 layer
// output; else residual + output in fp32
PyObject* moe(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!want(n, 8)) return nullptr;
  const at::Tensor* x = plain_state() ? tensor(a[0]) : nullptr;
  if (!x || x->scalar_type() != at::kBFloat16 || x->dim() < 1 || !x->is_contiguous() || x->numel() == 0 ||
      !PyLong_CheckExact(a[3]))
    Py_RETURN_NONE;
  const at::Device device = x->device();
  const int64_t h = x->size(-1), t = x->numel() / h;
  dflash_w4 gu, dn, sgu, sdn;
  if (!bank(a[1], 3, device, &gu) || !bank(a[2], 3, device, &dn)) Py_RETURN_NONE;
  const long k = PyLong_AsLong(a[3]);
  if (k < 1 || k > gu.experts) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const int64_t e = gu.experts;
  const at::Tensor* router = exactly(a[4], at::kBFloat16, {e, h}, device);
  if (!router) Py_RETURN_NONE;
  const at::Tensor* gate = nullptr;
  const bool shared = a[5] != Py_None;
  if (shared) {
    if (Py_TYPE(a[5]) != g_shared_type || !bank(PyTuple_GET_ITEM(a[5], 0), 2, device, &sgu) ||
        !bank(PyTuple_GET_ITEM(a[5], 1), 2, device, &sdn))
      Py_RETURN_NONE;
    gate = tensor(PyTuple_GET_ITEM(a[5], 2));
    if (!gate || gate->scalar_type() != at::kBFloat16 || gate->device() != device || gate->numel() != h || !gate->is_contiguous())
      Py_RETURN_NONE;
  }
  const at::Tensor* residual = nullptr;
  if (a[7] != Py_None && (!(residual = exactly(a[7], at::kFloat, {t, h}, device)) || tracked(*residual))) Py_RETURN_NONE;
  at::Tensor ws;
  const size_t need = g_entry.moe_workspace_bytes(t, h, gu.rows / 2, e, k, gu.group_size, shared);
  if (!workspace_of(a[6], need, device, &ws)) Py_RETURN_NONE;
  at::Tensor out = make({t, h}, residual ? at::kFloat : at::kBFloat16, device);
  // the routing outputs, which the plain call does not return: one block, each part 256-byte aligned
  const auto part = [](int64_t words) { return (words + 63) / 64 * 64; };
  const at::Tensor routing = make({part(t * e) + 4 * part(t * k) + part(e + 1)}, at::kInt, device);
  int32_t* logits = static_cast<int32_t*>(routing.data_ptr());
  int32_t *ids = logits + part(t * e), *wts = ids + part(t * k), *perm = wts + part(t * k), *inv = perm + part(t * k),
          *offsets = inv + part(t * k);
  const dflash_w4 *pu = shared ? &sgu : nullptr, *pd = shared ? &sdn : nullptr;
  const void* pg = shared ? gate->data_ptr() : nullptr;
  void* st = stream_of(device);
  int status;
  Py_BEGIN_ALLOW_THREADS
  if (residual)
    status = g_entry.moe_residual(x->data_ptr(), t, h, router->data_ptr(), k, &gu, &dn, pu, pd, pg,
                                  static_cast<const float*>(residual->data_ptr()), static_cast<float*>(out.data_ptr()),
                                  reinterpret_cast<float*>(logits), ids, reinterpret_cast<float*>(wts), perm, inv, offsets,
                                  ws.data_ptr(), ws.numel(), st);
  else
    status = g_entry.moe(x->data_ptr(), t, h, nullptr, router->data_ptr(), k, &gu, &dn, pu, pd, pg, out.data_ptr(),
                         reinterpret_cast<float*>(logits), ids, reinterpret_cast<float*>(wts), perm, inv, offsets,
                         ws.data_ptr(), ws.numel(), st);
  Py_END_ALLOW_THREADS
  if (status) return refused(residual ? "dflash_moe_w4a16_residual" : "dflash_moe_w4a16", status);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// ops._residual
const at::Tensor* residual_stream(PyObject* o) {
  const at::Tensor* t = plain_state() ? tensor(o) : nullptr;
  if (!t || t->dim() != 2 || !exactly(o, at::kFloat, t->sizes(), t->device()) || t->size(0) < 1 || t->size(0) > 1 << 19 ||
      t->size(1) % 512 || t->size(1) < 512 || t->size(1) > 8192 || tracked(*t))
    return nullptr;
  return t;
}

bool matrix(PyObject* o, int64_t rows, int64_t cols, at::Device device, dflash_w4* d) {
  return bank(o, 2, device, d) && d->rows == rows && d->cols == cols;
}

// gdn(hidden, history, state, in_proj, out_proj, input_norm, post_norm, norm, a_log, dt_bias, conv, key_heads, eps):
// the fields of ops.GdnMixer
PyObject* gdn(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!want(n, 13)) return nullptr;
  const at::Tensor* x = residual_stream(a[0]);
  const at::Tensor* a_log = x ? tensor(a[8]) : nullptr;
  if (!a_log || a_log->dim() != 1 || !PyLong_CheckExact(a[11]) || !PyFloat_CheckExact(a[12])) Py_RETURN_NONE;
  const at::Device device = x->device();
  const int64_t t = x->size(0), h = x->size(1), hv = a_log->size(0), hk = PyLong_AsLong(a[11]);
  if (hk < 1 || hk > 1024 || hv < 1 || hv > 1024 || hv % hk) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const int64_t width = 128 * (2 * hk + hv);
  const at::Tensor *history = exactly(a[1], at::kBFloat16, {1, width, 3}, device),
                   *state = exactly(a[2], at::kFloat, {1, hv, 128, 128}, device),
                   *input_norm = exactly(a[5], at::kFloat, {h}, device), *post_norm = exactly(a[6], at::kFloat, {h}, device),
                   *norm = exactly(a[7], at::kFloat, {128}, device), *dt_bias = exactly(a[9], at::kFloat, {hv}, device),
                   *conv = exactly(a[10], at::kBFloat16, {width, 1, 4}, device);
  dflash_gdn g{};
  if (!history || !state || !input_norm || !post_norm || !norm || !dt_bias || !conv ||
      tracked(*history) || tracked(*state) || tracked(*input_norm) || tracked(*post_norm) || tracked(*norm) ||
      tracked(*dt_bias) || tracked(*conv) || tracked(*a_log) || !exactly(a[8], at::kFloat, {hv}, device) ||
      !matrix(a[3], width + 128 * hv + 2 * hv, h, device, &g.in_proj) || !matrix(a[4], h, 128 * hv, device, &g.out_proj))
    Py_RETURN_NONE;
  g.input_norm = static_cast<const float*>(input_norm->data_ptr());
  g.post_norm = static_cast<const float*>(post_norm->data_ptr());
  g.norm = static_cast<const float*>(norm->data_ptr());
  g.a_log = static_cast<const float*>(a_log->data_ptr());
  g.dt_bias = static_cast<const float*>(dt_bias->data_ptr());
  g.conv = conv->data_ptr();
  g.hidden_size = h;
  g.key_heads = hk;
  g.value_heads = hv;
  g.eps = static_cast<float>(PyFloat_AS_DOUBLE(a[12]));
  at::Tensor o[9] = {make({t, h}, at::kFloat, device), make({t, h}, at::kBFloat16, device),
                     make({1, width, 3 + t}, at::kBFloat16, device), make({1, width, 3}, at::kBFloat16, device),
                     make({(t + 15) / 16, 1, hv, 128, 128}, at::kFloat, device),
                     make({1, hv, t, 128}, at::kFloat, device), make({1, hv, t, 128}, at::kFloat, device),
                     make({1, hv, t}, at::kFloat, device), make({1, hv, t, 128}, at::kFloat, device)};
  const auto f = [&](int i) { return static_cast<float*>(o[i].data_ptr()); };
  const at::Tensor ws = bytes(g_entry.gdn_workspace_bytes(t, h, hk, hv), device);
  void* st = stream_of(device);
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = g_entry.gdn(&g, static_cast<const float*>(x->data_ptr()), t, history->data_ptr(),
                       static_cast<const float*>(state->data_ptr()), f(0), o[1].data_ptr(), o[2].data_ptr(), o[3].data_ptr(), f(4),
                       f(5), f(6), f(7), f(8), ws.data_ptr(), ws.numel(), st);
  Py_END_ALLOW_THREADS
  if (status) return refused("dflash_gdn_mixer", status);
  PyObject* r = PyTuple_New(9);
  for (int i = 0; r && i < 9; ++i) PyTuple_SET_ITEM(r, i, THPVariable_Wrap(std::move(o[i])));
  return r;
  END_HANDLE_TH_ERRORS
}

// rms_norm(hidden, weight, eps)
PyObject* rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!want(n, 3)) return nullptr;
  const at::Tensor* x = residual_stream(a[0]);
  const at::Tensor* w = x ? exactly(a[1], at::kFloat, {x->size(1)}, x->device()) : nullptr;
  if (!w || !PyFloat_CheckExact(a[2]) || tracked(*w)) Py_RETURN_NONE;
  at::Tensor out = make(x->sizes(), at::kFloat, x->device());
  void* st = stream_of(x->device());
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = g_entry.rms_norm(static_cast<const float*>(x->data_ptr()), x->size(0), x->size(1),
                            static_cast<const float*>(w->data_ptr()), static_cast<float>(PyFloat_AS_DOUBLE(a[2])),
                            static_cast<float*>(out.data_ptr()), st);
  Py_END_ALLOW_THREADS
  if (status) return refused("dflash_rms_norm", status);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// attention(hidden, keys, values, position, in_proj, out_proj, input_norm, post_norm, q_norm, k_norm, inv_freq, heads,
// kv_heads, head_dim, eps): (mid, normed)
PyObject* attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!want(n, 15)) return nullptr;
  const at::Tensor* x = residual_stream(a[0]);
  const at::Tensor *keys = x ? tensor(a[1]) : nullptr, *inv_freq = x ? tensor(a[10]) : nullptr;
  if (!keys || keys->dim() != 4 || keys->size(2) > 1 << 24 || !inv_freq || inv_freq->dim() != 1 ||
      !PyFloat_CheckExact(a[14]))
    Py_RETURN_NONE;
  int64_t v[4];
  const int at_[4] = {3, 11, 12, 13};
  for (int i = 0; i < 4; ++i) {
    if (!PyLong_CheckExact(a[at_[i]])) Py_RETURN_NONE;
    v[i] = PyLong_AsLong(a[at_[i]]);
    if (v[i] < 0 || v[i] > 1 << 24) {
      PyErr_Clear();
      Py_RETURN_NONE;
    }
  }
  const at::Device device = x->device();
  const int64_t t = x->size(0), h = x->size(1), position = v[0], heads = v[1], kv = v[2], d = v[3], half = inv_freq->size(0);
  if ((d != 128 && d != 256) || kv < 1 || heads < 1 || heads > 1024 || heads % kv || t * heads > 1 << 22 ||
      position + t > keys->size(2) || half < 1 || half % (d / 64) || 2 * half > d)
    Py_RETURN_NONE;
  const int64_t cache[4] = {1, kv, keys->size(2), d};
  const at::Tensor *values = exactly(a[2], at::kBFloat16, cache, device),
                   *input_norm = exactly(a[6], at::kFloat, {h}, device), *post_norm = exactly(a[7], at::kFloat, {h}, device),
                   *q_norm = exactly(a[8], at::kFloat, {d}, device), *k_norm = exactly(a[9], at::kFloat, {d}, device);
  dflash_attention g{};
  if (!exactly(a[1], at::kBFloat16, cache, device) || !values || !input_norm || !post_norm || !q_norm || !k_norm ||
      tracked(*keys) || tracked(*values) || tracked(*input_norm) || tracked(*post_norm) || tracked(*q_norm) ||
      tracked(*k_norm) || tracked(*inv_freq) || !exactly(a[10], at::kFloat, {half}, device) ||
      !matrix(a[4], 2 * (heads + kv) * d, h, device, &g.in_proj) || !matrix(a[5], h, heads * d, device, &g.out_proj))
    Py_RETURN_NONE;
  g.input_norm = static_cast<const float*>(input_norm->data_ptr());
  g.post_norm = static_cast<const float*>(post_norm->data_ptr());
  g.q_norm = static_cast<const float*>(q_norm->data_ptr());
  g.k_norm = static_cast<const float*>(k_norm->data_ptr());
  g.inv_freq = static_cast<const float*>(inv_freq->data_ptr());
  g.hidden_size = h;
  g.heads = heads;
  g.kv_heads = kv;
  g.head_dim = d;
  g.rotary_dim = 2 * half;
  g.eps = static_cast<float>(PyFloat_AS_DOUBLE(a[14]));
  at::Tensor mid = make({t, h}, at::kFloat, device), normed = make({t, h}, at::kBFloat16, device);
  const at::Tensor ws = bytes(g_entry.attention_workspace_bytes(t, h, heads, kv, d), device);
  void* st = stream_of(device);
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = g_entry.attention(&g, static_cast<const float*>(x->data_ptr()), t, position, keys->data_ptr(), values->data_ptr(),
                             keys->size(2), static_cast<float*>(mid.data_ptr()), normed.data_ptr(), ws.data_ptr(), ws.numel(), st);
  Py_END_ALLOW_THREADS
  if (status) return refused("dflash_attention_mixer", status);
  PyObject* r = PyTuple_New(2);
  if (r) {
    PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(std::move(mid)));
    PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(std::move(normed)));
  }
  return r;
  END_HANDLE_TH_ERRORS
}

// commit(state, keys, u, cum, accepted, window, first): (state, history), as ops.gdn_commit
PyObject* commit(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!want(n, 7)) return nullptr;
  const at::Tensor* state = plain_state() ? tensor(a[0]) : nullptr;
  const at::Tensor *keys = tensor(a[1]), *u = tensor(a[2]), *cum = tensor(a[3]), *window = tensor(a[5]);
  if (!state || !keys || !u || !cum || !window || !PyLong_CheckExact(a[4]) || !PyLong_CheckExact(a[6]) || state->dim() != 4)
    Py_RETURN_NONE;
  const int64_t j = PyLong_AsLong(a[4]), first = PyLong_AsLong(a[6]), hv = state->size(1);
  const at::Device device = state->device();
  const auto f32 = [&](const at::Tensor* t) { return t->scalar_type() == at::kFloat && t->device() == device; };
  if (j < 1 || j > 16 || first < 0 || first > 1 << 24 || hv > 1024 ||
      !exactly(a[0], at::kFloat, {1, hv, 128, 128}, device) || keys->dim() != 4 || keys->size(0) != 1 ||
      keys->size(1) != hv || keys->size(2) < j || keys->size(3) != 128 || u->sizes() != keys->sizes() ||
      cum->sizes() != keys->sizes().slice(0, 3) || !f32(keys) || !f32(u) || !f32(cum) || keys->stride(2) != 128 ||
      keys->stride(3) != 1 || u->strides() != keys->strides() || cum->stride(2) != 1 ||
      window->scalar_type() != at::kBFloat16 || window->dim() != 3 || window->size(0) != 1 || window->device() != device ||
      !window->is_contiguous() || first + 3 > window->size(2) || tracked(*state) || tracked(*keys) || tracked(*u) ||
      tracked(*cum) || tracked(*window)) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  at::Tensor out = make(state->sizes(), at::kFloat, device), history = make({1, window->size(1), 3}, at::kBFloat16, device);
  const auto f = [](const at::Tensor* t) { return static_cast<const float*>(t->data_ptr()); };
  void* st = stream_of(device);
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = g_entry.commit(f(state), f(keys), f(u), f(cum), keys->stride(1), cum->stride(1), hv, j,
                          static_cast<float*>(out.data_ptr()), window->data_ptr(), window->size(2), first, window->size(1),
                          history.data_ptr(), st);
  Py_END_ALLOW_THREADS
  if (status) return refused("dflash_gdn_commit", status);
  PyObject* r = PyTuple_New(2);
  if (r) {
    PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(std::move(out)));
    PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(std::move(history)));
  }
  return r;
  END_HANDLE_TH_ERRORS
}

// bind(PackedW4, SharedExpert, _lib.check, address of an entry by name)
PyObject* bind(PyObject*, PyObject* args) {
  PyObject *packed, *shared, *check, *find;
  if (!PyArg_ParseTuple(args, "O!O!OO", &PyType_Type, &packed, &PyType_Type, &shared, &check, &find)) return nullptr;
  bool ok = true;
  const auto get = [&](const char* name, auto& fn) {
    PyObject* v = ok ? PyObject_CallFunction(find, "s", name) : nullptr;
    void* p = v ? PyLong_AsVoidPtr(v) : nullptr;
    Py_XDECREF(v);
    ok = ok && p && !PyErr_Occurred();
    fn = reinterpret_cast<std::decay_t<decltype(fn)>>(p);
  };
  get("dflash_qlinear_workspace_bytes", g_entry.qlinear_workspace_bytes);
  get("dflash_qlinear_w4a16", g_entry.qlinear);
  get("dflash_qlinear_w4a16_f32", g_entry.qlinear_f32);
  get("dflash_moe_workspace_bytes", g_entry.moe_workspace_bytes);
  get("dflash_moe_w4a16", g_entry.moe);
  get("dflash_moe_w4a16_residual", g_entry.moe_residual);
  get("dflash_gdn_workspace_bytes", g_entry.gdn_workspace_bytes);
  get("dflash_gdn_mixer", g_entry.gdn);
  get("dflash_gdn_commit", g_entry.commit);
  get("dflash_rms_norm", g_entry.rms_norm);
  get("dflash_attention_workspace_bytes", g_entry.attention_workspace_bytes);
  get("dflash_attention_mixer", g_entry.attention);
  if (!ok) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "bind: an entry has no address");
    return nullptr;
  }
  Py_INCREF(packed);
  Py_INCREF(shared);
  Py_INCREF(check);
  g_check = check;
  g_packed_type = reinterpret_cast<PyTypeObject*>(packed);
  g_shared_type = reinterpret_cast<PyTypeObject*>(shared);
  Py_RETURN_NONE;
}

#define FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST(linear), FAST(moe), FAST(gdn), FAST(attention), FAST(commit), FAST(rms_norm),
                         {"bind", bind, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "dflash_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_dflash_host() {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "TORCH", DFLASH_TORCH) < 0) Py_CLEAR(m);  // the torch it was compiled for
  return m;
}
