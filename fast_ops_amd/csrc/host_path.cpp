// The host's share of an attention call, in C++: what flash_attention.py does between its arguments and the C entry points - sizes and
// strides out of the tensors, outputs and scratch memory allocated, the call itself - for the calls that need nothing else. Whatever
// is not plainly one of those (other types, shapes, layouts, devices; tensor subclasses; torch's modes and transforms; a backward whose
// workspace finds no memory) is declined with None, and the Python code does it, or refuses it, as it always has. Outputs that find no
// memory raise torch.OutOfMemoryError from here. Nothing is kept between calls but what a thread was last refused (Refusal).
//
// Why: a short call is its host time. B=2 H=4 S=128 at head_dim 64, without gradients 9.5 -> 4.7 us of it, of which the launch takes about 2.5
// and two allocations 1.2; forward and backward 112 -> 77 us (the rest is autograd's: a product by a number takes 42 there).
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>

#include <cmath>

#include "../../include/fastops.h"

namespace {

bool ready = false;
decltype(&fo_attn_fwd_ex_ws) p_fwd_ex_ws;
decltype(&fo_attn_fwd_workspace_ex) p_fwd_workspace;
decltype(&fo_attn_bwd_ws) p_bwd_ws;
decltype(&fo_attn_bwd_workspace_ex) p_bwd_workspace;
decltype(&fo_strerror) p_strerror;
PyObject* current_device = nullptr;      // torch's functions of these names
PyObject* raw_stream = nullptr;

// Scratch memory that a thread was refused: the next kRetry calls that would ask for as much or more on that device do not (a request
// that fails makes the caching allocator give its cached blocks back, and the calls after it allocate anew).
constexpr int kRetry = 256;
struct Refusal {
  int64_t bytes = 0;
  int device = -1, calls = 0;
  bool covers(int dev, int64_t n) {
    if (calls == 0 || dev != device || n < bytes) return false;
    --calls;
    return true;
  }
  void note(int dev, int64_t n) { bytes = n; device = dev; calls = kRetry; }
};
thread_local Refusal refused_fwd, refused_bwd;

struct Dims { int64_t B, H, Sq, Sk, D; };

bool plain_mode() {
  return !c10::impl::dispatch_mode_enabled() && !at::impl::torch_function_mode_enabled() &&
         !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
         !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Python);
}

// an ordinary dense GPU tensor (its autograd keys aside), as an exact torch.Tensor or Parameter
bool plain(PyObject* o, const at::Tensor*& t) {
  if (!THPVariable_CheckExact(o)) return false;
  t = &THPVariable_Unpack(o);
  static const c10::DispatchKeySet ordinary = c10::DispatchKeySet(c10::DispatchKey::CUDA) | c10::autograd_dispatch_keyset |
                                              c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView) | c10::autocast_dispatch_keyset;
  return t->defined() && t->is_cuda() && t->layout() == at::kStrided && !t->is_neg() && !t->is_conj() && (t->key_set().raw_repr() & ~(ordinary.raw_repr() | c10::full_backend_mask)) == 0 &&
         !t->unsafeGetTensorImpl()->has_symbolic_sizes_strides() && !t->_fw_grad(0).defined();
}

bool operands(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, bool bshd, Dims& d) {
  if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4) return false;
  const auto type = q.scalar_type();
  if ((type != at::kHalf && type != at::kBFloat16) || k.scalar_type() != type || v.scalar_type() != type) return false;
  if (k.get_device() != q.get_device() || v.get_device() != q.get_device()) return false;
  if (q.stride(3) != 1 || k.stride(3) != 1 || v.stride(3) != 1) return false;
  const int h = bshd ? 2 : 1, s = bshd ? 1 : 2;
  d = {q.size(0), q.size(h), q.size(s), k.size(s), q.size(3)};
  if (k.size(0) != d.B || k.size(h) != d.H || k.size(3) != d.D || v.sizes() != k.sizes()) return false;
  constexpr int64_t most = 0x7FFFFFFF;
  return d.D <= 128 && d.D % 8 == 0 && d.D > 0 && d.B > 0 && d.H > 0 && d.Sq > 0 && d.Sk > 0 && d.B <= most && d.H <= most && d.Sq <= most && d.Sk <= most;
}

void strides_of(const at::Tensor& t, bool bshd, int64_t* out) {
  out[0] = t.stride(0);
  out[1] = t.stride(bshd ? 2 : 1);
  out[2] = t.stride(bshd ? 1 : 2);
}

// dropout: None or (p, seed, offset); bias: None or [B|1, H|1, Sq|1, Sk]. False: declined.
bool extras_of(PyObject* dropout, PyObject* bias, const at::Tensor& q, const Dims& d, fo_attn_extras& ex, bool& any) {
  ex = fo_attn_extras{};
  any = false;
  if (bias != Py_None) {
    const at::Tensor* b;
    if (!plain(bias, b) || b->dim() != 4 || b->get_device() != q.get_device() || b->stride(3) != 1) return false;
    if (b->scalar_type() != q.scalar_type() && b->scalar_type() != at::kFloat) return false;
    const int64_t want[4] = {d.B, d.H, d.Sq, d.Sk};
    for (int i = 0; i < 3; ++i) {
      if (b->size(i) != want[i] && b->size(i) != 1) return false;
      ex.bias_strides[i] = b->size(i) == 1 && want[i] != 1 ? 0 : b->stride(i);      // (as Tensor.expand has them)
    }
    if (b->size(3) != d.Sk) return false;
    ex.bias = b->data_ptr();
    ex.bias_dtype = b->scalar_type() == at::kFloat ? FO_DTYPE_F32 : b->scalar_type() == at::kHalf ? FO_DTYPE_F16 : FO_DTYPE_BF16;
    any = true;
  }
  if (dropout != Py_None) {
    if (!PyTuple_CheckExact(dropout) || PyTuple_GET_SIZE(dropout) != 3) return false;
    PyObject *p = PyTuple_GET_ITEM(dropout, 0), *seed = PyTuple_GET_ITEM(dropout, 1), *offset = PyTuple_GET_ITEM(dropout, 2);
    if (!PyFloat_CheckExact(p) || !PyLong_CheckExact(seed) || !PyLong_CheckExact(offset)) return false;
    if (PyFloat_AS_DOUBLE(p) != 0.0) {
      ex.dropout_p = (float)PyFloat_AS_DOUBLE(p);
      ex.dropout_seed = (uint32_t)PyLong_AsUnsignedLongLongMask(seed);
      ex.dropout_offset = PyLong_AsUnsignedLongLongMask(offset);
      any = true;
    }
  }
  return true;
}

// the raw stream that is current on the tensors' device, if that device is the current one
bool stream_on(int64_t device, void*& stream) {
  PyObject* now = PyObject_CallNoArgs(current_device);
  if (now == nullptr) return false;
  const long at = PyLong_AsLong(now);
  Py_DECREF(now);
  if (at != device) return false;
  PyObject* index = PyLong_FromLong(at);
  PyObject* raw = PyObject_CallOneArg(raw_stream, index);
  Py_DECREF(index);
  if (raw == nullptr) return false;
  stream = (void*)(uintptr_t)PyLong_AsUnsignedLongLongMask(raw);
  Py_DECREF(raw);
  return true;
}

PyObject* declined() {
  PyErr_Clear();
  Py_RETURN_NONE;
}
PyObject* failed(const char* what, int status) {
  return PyErr_Format(PyExc_RuntimeError, "%s: %s (fo_status %d)", what, p_strerror(status), status);
}
bool scale_of(PyObject* o, int64_t D, float& scale) {
  if (o == Py_None) { scale = (float)(1.0 / std::sqrt((double)D)); return true; }
  if (!PyFloat_CheckExact(o)) return false;
  const double s = PyFloat_AS_DOUBLE(o);
  scale = (float)(s != 0.0 ? s : 1.0 / std::sqrt((double)D));
  return true;
}

// fwd(q, k, v, bshd, causal, scale or None, dropout or None, bias or None) -> (o, lse) or None
PyObject* fwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
  const at::Tensor *q, *k, *v;
  Dims d;
  fo_attn_extras ex;
  bool any;
  float scale;
  void* stream;
  int status = 0;
  at::Tensor o, lse;
  HANDLE_TH_ERRORS
  if (n != 8 || !ready || !plain_mode() || !plain(a[0], q) || !plain(a[1], k) || !plain(a[2], v)) return declined();
  if (!PyBool_Check(a[3]) || !PyBool_Check(a[4])) return declined();
  const bool bshd = a[3] == Py_True, causal = a[4] == Py_True;
  if (!operands(*q, *k, *v, bshd, d) || !scale_of(a[5], d.D, scale) || !extras_of(a[6], a[7], *q, d, ex, any) || !stream_on(q->get_device(), stream)) return declined();
  {
    pybind11::gil_scoped_release no_gil;
    int64_t qs[3], ks[3], vs[3], os[3];
    strides_of(*q, bshd, qs); strides_of(*k, bshd, ks); strides_of(*v, bshd, vs);
    // (a layout that empty_like keeps; anything else gets a plain contiguous output)
    o = at::empty_like(*q);
    if (o.strides() != q->strides()) o = at::empty(q->sizes(), q->options());
    lse = at::empty({d.B, d.H, d.Sq}, q->options().dtype(at::kFloat));
    strides_of(o, bshd, os);
    const int type = q->scalar_type() == at::kHalf ? FO_DTYPE_F16 : FO_DTYPE_BF16;
    const int64_t bytes = p_fwd_workspace((int)d.B, (int)d.H, (int)d.Sq, (int)d.Sk, (int)d.D, ks, vs, causal, any ? &ex : nullptr);
    at::Tensor ws;
    void* room = nullptr;
    if (bytes > 0 && !refused_fwd.covers((int)q->get_device(), bytes)) {
      try {
        ws = at::empty({bytes}, q->options().dtype(at::kByte));
        room = ws.data_ptr();
      } catch (const c10::OutOfMemoryError&) {      // (the call does without)
        refused_fwd.note((int)q->get_device(), bytes);
      }
    }
    status = p_fwd_ex_ws(q->data_ptr(), k->data_ptr(), v->data_ptr(), o.data_ptr(), (float*)lse.data_ptr(), (int)d.B, (int)d.H, (int)d.Sq, (int)d.Sk, (int)d.D,
                         qs, ks, vs, os, scale, causal, type, any ? &ex : nullptr, room, room != nullptr ? bytes : 0, stream);
  }
  if (status != 0) return failed("fo_attn_fwd", status);
  PyObject *po = THPVariable_Wrap(std::move(o)), *pl = THPVariable_Wrap(std::move(lse));
  PyObject* both = PyTuple_Pack(2, po, pl);
  Py_DECREF(po);
  Py_DECREF(pl);
  return both;
  END_HANDLE_TH_ERRORS
}

// bwd(q, k, v, o, lse, d_o, bshd, causal, scale or None, dropout or None, bias or None) -> (dq, dk, dv) or None
PyObject* bwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
  const at::Tensor *q, *k, *v, *o, *lse, *g;
  Dims d;
  fo_attn_extras ex;
  bool any, room = true;
  float scale;
  void* stream;
  int status = 0;
  at::Tensor dq, dk, dv;
  HANDLE_TH_ERRORS
  if (n != 11 || !ready || !plain_mode()) return declined();
  if (!plain(a[0], q) || !plain(a[1], k) || !plain(a[2], v) || !plain(a[3], o) || !plain(a[4], lse) || !plain(a[5], g)) return declined();
  if (!PyBool_Check(a[6]) || !PyBool_Check(a[7])) return declined();
  const bool bshd = a[6] == Py_True, causal = a[7] == Py_True;
  if (!operands(*q, *k, *v, bshd, d) || !scale_of(a[8], d.D, scale) || !extras_of(a[9], a[10], *q, d, ex, any)) return declined();
  if (g->scalar_type() != q->scalar_type() || g->sizes() != q->sizes() || o->scalar_type() != q->scalar_type() || o->sizes() != q->sizes()) return declined();
  if (o->stride(3) != 1 || g->stride(3) != 1 || o->get_device() != q->get_device() || g->get_device() != q->get_device()) return declined();
  for (int i = 0; i < 3 && !g->is_contiguous(); ++i)
    if (g->stride(i) % 8 != 0) return declined();
  if (lse->scalar_type() != at::kFloat || !lse->is_contiguous() || lse->numel() != d.B * d.H * d.Sq || lse->get_device() != q->get_device()) return declined();
  if (!stream_on(q->get_device(), stream)) return declined();
  const int64_t bytes = p_bwd_workspace((int)d.B, (int)d.H, (int)d.Sq, (int)d.Sk, (int)d.D, causal, any ? &ex : nullptr);
  if (refused_bwd.covers((int)q->get_device(), bytes)) return declined();      // (the Python code keeps to a smaller one for as long)
  {
    pybind11::gil_scoped_release no_gil;
    dq = at::empty(q->sizes(), q->options());
    dk = at::empty(k->sizes(), q->options());
    dv = at::empty(v->sizes(), q->options());
    const int type = q->scalar_type() == at::kHalf ? FO_DTYPE_F16 : FO_DTYPE_BF16;
    at::Tensor ws;
    try {
      ws = at::empty({bytes}, q->options().dtype(at::kByte));
    } catch (const c10::OutOfMemoryError&) {
      room = false;
    }
    if (room) {
      int64_t st[8][3];
      const int64_t* list[8];
      const at::Tensor* ts[8] = {q, k, v, o, g, &dq, &dk, &dv};
      for (int i = 0; i < 8; ++i) { strides_of(*ts[i], bshd, st[i]); list[i] = st[i]; }
      status = p_bwd_ws(q->data_ptr(), k->data_ptr(), v->data_ptr(), o->data_ptr(), g->data_ptr(), (const float*)lse->data_ptr(), dq.data_ptr(), dk.data_ptr(),
                        dv.data_ptr(), (int)d.B, (int)d.H, (int)d.Sq, (int)d.Sk, (int)d.D, list, scale, causal, type, any ? &ex : nullptr, ws.data_ptr(), bytes, stream);
    }
  }
  if (!room) { refused_bwd.note((int)q->get_device(), bytes); return declined(); }
  if (status != 0) return failed("fo_attn_bwd_ws", status);
  PyObject *pq = THPVariable_Wrap(std::move(dq)), *pk = THPVariable_Wrap(std::move(dk)), *pv = THPVariable_Wrap(std::move(dv));
  PyObject* all = PyTuple_Pack(3, pq, pk, pv);
  Py_DECREF(pq);
  Py_DECREF(pk);
  Py_DECREF(pv);
  return all;
  END_HANDLE_TH_ERRORS
}

// init({name: address of the entry point}, torch._C._cuda_getDevice, torch._C._cuda_getCurrentRawStream)
PyObject* init(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 3 || !PyDict_Check(a[0])) return PyErr_Format(PyExc_TypeError, "init(addresses, current_device, raw_stream)");
  auto address = [&](const char* name) -> void* {
    PyObject* at = PyDict_GetItemString(a[0], name);
    return at != nullptr ? (void*)(uintptr_t)PyLong_AsUnsignedLongLongMask(at) : nullptr;
  };
  p_fwd_ex_ws = (decltype(p_fwd_ex_ws))address("fo_attn_fwd_ex_ws");
  p_fwd_workspace = (decltype(p_fwd_workspace))address("fo_attn_fwd_workspace_ex");
  p_bwd_ws = (decltype(p_bwd_ws))address("fo_attn_bwd_ws");
  p_bwd_workspace = (decltype(p_bwd_workspace))address("fo_attn_bwd_workspace_ex");
  p_strerror = (decltype(p_strerror))address("fo_strerror");
  Py_INCREF(a[1]);
  Py_INCREF(a[2]);
  current_device = a[1];
  raw_stream = a[2];
  ready = p_fwd_ex_ws && p_fwd_workspace && p_bwd_ws && p_bwd_workspace && p_strerror;
  return PyBool_FromLong(ready);
}

PyMethodDef methods[] = {{"fwd", (PyCFunction)(void (*)())fwd, METH_FASTCALL, nullptr},
                         {"bwd", (PyCFunction)(void (*)())bwd, METH_FASTCALL, nullptr},
                         {"init", (PyCFunction)(void (*)())init, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "the host's share of an attention call", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&module); }
