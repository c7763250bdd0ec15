// The host side of the calls that a network makes once per layer, for the Python front end: what backend.conv_forward,
// dense_forward, bn_forward, bn_backward and conv_wgrad do in the usual case, from tensors to the library's entry point,
// without the interpreter in between.  A layer costs the host its launch (3 us) and the output's allocation (1 us); the checks,
// pointer reads and argument conversions in Python and ctypes cost 6 us beside them (a norm's 12), more than half the time of
// the kernel of a small layer: one 16 -> 16 layer on 21 k rows 16.9 us a call, 11.8 this way.
//
// Nothing is decided here: the caller passes the dataflow and the map's arrays as tensors.  What is not the usual call (other
// layouts, dtypes, devices, wrapped tensors, anything that has to be refused) is answered with None, and the caller's general
// path takes it, copies where it must and words the errors.  No state is kept.
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Exceptions.h>
#include <ATen/ATen.h>

#include "pcengine_amd.h"

// entry points that a library beside this extension may be without, as the stubs are that its host side is tested beside (the library
// that the package loads has all of them, or is refused): the calls that need them are then declined
#pragma weak pce_bn_forward_counted
#pragma weak pce_bn_backward_masked
#pragma weak pce_conv_wgrad_add

namespace {

enum Kind { KIND_OSO = 0, KIND_OSB = 1, KIND_OS = 2, KIND_FDS = 3, KIND_DENSE = 4 };

// Other Python threads run while a call allocates or launches (both may wait for the device), as they do around a ctypes call.
struct Unlocked {
  PyThreadState *state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
  Unlocked(const Unlocked &) = delete;
  Unlocked() = default;
};

// a plain tensor on a GPU: not one that stands for another (functorch, fake tensors and other modes)
const at::Tensor *plain(PyObject *o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor &t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || !t.has_storage() || t.layout() != at::kStrided || t.is_neg() || t.is_conj() ||
      t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                               c10::DispatchKey::Functionalize, c10::DispatchKey::ZeroTensor})))
    return nullptr;
  return &t;
}

// elements between rows the kernels can use in place: 0 dense, -1 neither (backend._row_stride)
int64_t row_stride(const at::Tensor &t) {
  if (t.is_contiguous()) return 0;
  const int64_t ld = t.stride(0), c = t.size(1);
  return t.stride(1) == 1 && ld > c && ld % 8 == 0 && c % 8 == 0 && (uintptr_t)t.data_ptr() % 16 == 0 ? ld : -1;
}

struct View {   // the integers and arrays of a map, as the caller laid them out for the kind of layer
  PyObject *tuple;
  bool bad = false;
  int64_t num(Py_ssize_t i) const { return PyLong_AsLongLong(PyTuple_GET_ITEM(tuple, i)); }
  const int32_t *array(Py_ssize_t i, const at::Device &dev) {
    PyObject *o = PyTuple_GET_ITEM(tuple, i);
    if (o == Py_None) return nullptr;
    const at::Tensor *t = plain(o);
    if (!t || t->scalar_type() != at::kInt || t->device() != dev || !t->is_contiguous()) {
      bad = true;
      return nullptr;
    }
    return t->data_ptr<int32_t>();
  }
};

// the kv + 1 offsets that a map mirrors on the host, as the array the view holds: read at the call, never kept as an address
struct HostPos {
  Py_buffer buffer;
  bool held = false;
  const int32_t *read(PyObject *o, int64_t kv) {
    if (PyObject_GetBuffer(o, &buffer, PyBUF_SIMPLE)) {
      PyErr_Clear();
      return nullptr;
    }
    held = true;
    return buffer.len >= (Py_ssize_t)((kv + 1) * sizeof(int32_t)) ? (const int32_t *)buffer.buf : nullptr;
  }
  ~HostPos() {
    if (held) PyBuffer_Release(&buffer);
  }
};

// layer(kind, view, feats, weight, packed, bias, residual, out, act, slope, scratch, stream)
//   -> the output, or None where the general path has to take the call; an int is the library's error code
PyObject *layer(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 12 || !PyTuple_Check(args[1])) {
    PyErr_SetString(PyExc_TypeError, "layer: twelve arguments, the second one a tuple");
    return nullptr;
  }
  const long kind = PyLong_AsLong(args[0]);
  View v{args[1]};
  const at::Tensor *feats = plain(args[2]), *weight = plain(args[3]), *packed = nullptr, *scratch = nullptr;
  if (!feats || !weight || feats->dim() != 2 || !weight->is_contiguous()) Py_RETURN_NONE;
  const at::Device dev = feats->device();
  const auto dtype = feats->scalar_type();
  if ((dtype != at::kHalf && dtype != at::kFloat) || weight->scalar_type() != dtype || weight->device() != dev) Py_RETURN_NONE;
  const int dt = dtype == at::kHalf ? PCE_F16 : PCE_F32;
  const bool dense = kind == KIND_DENSE;
  if (weight->dim() != (dense ? 2 : 3)) Py_RETURN_NONE;
  const int64_t kv = dense ? 1 : weight->size(0), c_in = weight->size(-2), c_out = weight->size(-1);
  const int64_t n_in = dense ? feats->size(0) : v.num(0), n_out = dense ? n_in : v.num(1);
  if (feats->size(0) != n_in || feats->size(1) != c_in || (!dense && kv != v.num(2)) || n_in <= 0 || n_out <= 0 || c_in <= 0 || c_out <= 0)
    Py_RETURN_NONE;
  if (args[4] != Py_None) {
    packed = plain(args[4]);
    if (!packed || packed->device() != dev || !packed->is_contiguous()) Py_RETURN_NONE;
  }
  if (dt == PCE_F16 && !packed) Py_RETURN_NONE;
  pce_epilogue_t epi = {};
  epi.ld_in = row_stride(*feats);
  if (epi.ld_in < 0 || (dense && epi.ld_in)) Py_RETURN_NONE;
  if (args[5] != Py_None) {
    const at::Tensor *b = plain(args[5]);
    if (!b || b->scalar_type() != dtype || b->device() != dev || !b->is_contiguous() || b->numel() != c_out) Py_RETURN_NONE;
    epi.bias = b->data_ptr();
  }
  if (args[6] != Py_None) {
    const at::Tensor *r = plain(args[6]);
    if (!r || r->scalar_type() != dtype || r->device() != dev || !r->is_contiguous() || r->dim() != 2 || r->size(0) != n_out || r->size(1) != c_out)
      Py_RETURN_NONE;
    epi.residual = r->data_ptr();
  }
  epi.act = (int32_t)PyLong_AsLong(args[8]);
  epi.slope = (float)PyFloat_AsDouble(args[9]);
  at::Tensor made;
  const at::Tensor *out = nullptr;
  if (args[7] != Py_None) {
    out = plain(args[7]);
    if (!out || out->scalar_type() != dtype || out->device() != dev || out->dim() != 2 || out->size(0) != n_out || out->size(1) != c_out)
      Py_RETURN_NONE;
    epi.ld_out = row_stride(*out);
    if (epi.ld_out < 0 || (dense && epi.ld_out)) Py_RETURN_NONE;
  }
  if (args[10] != Py_None) {
    scratch = plain(args[10]);
    if (!scratch || scratch->device() != dev || !scratch->is_contiguous()) Py_RETURN_NONE;
  }
  // the arrays of the map, before anything is allocated
  const int32_t *m[8] = {};
  const int arrays = kind == KIND_OSO || kind == KIND_OSB ? 2 : kind == KIND_OS ? 1 : kind == KIND_FDS ? 7 : 0;
  for (int i = 0; i < arrays; ++i) m[i] = v.array(3 + i, dev);
  if (v.bad) Py_RETURN_NONE;
  HostPos kpos, qkpos;
  const int32_t *kpos_h = nullptr, *qkpos_h = nullptr;
  if (kind == KIND_FDS && (!(kpos_h = kpos.read(PyTuple_GET_ITEM(args[1], 13), kv)) || !(qkpos_h = qkpos.read(PyTuple_GET_ITEM(args[1], 14), kv))))
    Py_RETURN_NONE;
  void *stream = PyLong_AsVoidPtr(args[11]);
  if (PyErr_Occurred()) return nullptr;
  const void *x = feats->data_ptr(), *w = weight->data_ptr(), *wp = dt == PCE_F16 ? packed->data_ptr() : nullptr;
  if (kind == KIND_OSB) {   // the block kernel reads whole 16-byte pieces and addresses this many bytes of rows
    const uintptr_t all = (uintptr_t)x | (uintptr_t)wp | (uintptr_t)epi.bias | (uintptr_t)epi.residual | (out ? (uintptr_t)out->data_ptr() : 0);
    if (dt != PCE_F16 || all % 16 || n_in * (epi.ld_in ? epi.ld_in : c_in) * 2 >= 0xF0000000ll) Py_RETURN_NONE;
  }
  int64_t num[10] = {};   // the numbers behind n_in, n_out, kv and the arrays
  for (Py_ssize_t i = 3 + arrays; i < PyTuple_GET_SIZE(args[1]) && i < 3 + arrays + (kind == KIND_FDS ? 3 : 10); ++i) num[i - 3 - arrays] = v.num(i);
  if (PyErr_Occurred()) return nullptr;
  void *ws = scratch ? scratch->data_ptr() : nullptr;
  const int64_t ws_bytes = scratch ? (int64_t)scratch->nbytes() : 0;
  int rc = PCE_EINVAL;
  const int ci = (int)c_in, co = (int)c_out, k = (int)kv;
  {
    Unlocked unlocked;
    if (!out) {
      made = at::empty({n_out, c_out}, feats->options());
      out = &made;
    }
    void *y = out->data_ptr();
    const bool plain_call = !epi.bias && !epi.residual && epi.act == PCE_ACT_NONE && !epi.ld_in && !epi.ld_out;
    const pce_epilogue_t *e = plain_call ? nullptr : &epi;
    if (kind == KIND_OSO) {          // nbr, order | mid, heavy, nonzero, single
      rc = pce_conv_fwd_oso(x, w, wp, y, dt, n_in, n_out, ci, co, k, (int)num[0], m[0], m[1], num + 1, e, stream);
    } else if (kind == KIND_OSB) {   // nbr, order | pairs
      rc = pce_conv_fwd_osb(x, wp, y, dt, n_in, n_out, num[0], ci, co, k, m[0], m[1], ws, ws_bytes, e, stream);
    } else if (kind == KIND_OS) {    // nbr
      rc = ws ? pce_conv_fwd_os_parts(x, w, y, dt, n_in, n_out, ci, co, k, m[0], ws, ws_bytes, e, stream)
              : pce_conv_fwd_os(x, w, wp, y, dt, n_in, n_out, ci, co, k, m[0], e, stream);
    } else if (kind == KIND_FDS) {   // imap, omap, oslot, kpos, qkpos, ocsr, route | mid, pairs, qsum, kpos and qkpos on the host
      const int64_t es = dt == PCE_F16 ? 2 : 4;
      rc = pce_conv_fwd_fds(x, w, wp, y, dt, n_in, n_out, ci, co, k, (int)num[0], m[0], m[1], m[2], m[3], m[4], kpos_h, qkpos_h, m[5], m[6],
                            num[1], num[2], ws, ws ? ws_bytes / es : 0, e, stream);
    } else if (dense) {
      rc = pce_conv_fwd_dense(x, w, wp, y, dt, n_in, ci, co, e, stream);
    }
  }
  if (rc != PCE_OK) return PyLong_FromLong(rc);
  if (made.defined()) return THPVariable_Wrap(std::move(made));
  Py_INCREF(args[7]);
  return args[7];
  END_HANDLE_TH_ERRORS
}

// the [count] elements of `t` from element `from` on, as a tensor of their own in the same memory
at::Tensor part(const at::Tensor &t, int64_t from, int64_t count) {
  at::Tensor p = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(t.storage()), c10::DispatchKeySet(c10::DispatchKey::CUDA), t.dtype());
  p.unsafeGetTensorImpl()->set_storage_offset(t.storage_offset() + from);
  p.unsafeGetTensorImpl()->set_sizes_contiguous({count});
  return p;
}

// a dense vector of n floats, or nothing (allowed where `none` is)
bool floats(PyObject *o, const at::Device &dev, int64_t n, const float **p) {
  *p = nullptr;
  if (o == Py_None) return true;
  const at::Tensor *t = plain(o);
  if (!t || t->scalar_type() != at::kFloat || t->device() != dev || !t->is_contiguous() || t->numel() != n) return false;
  *p = t->data_ptr<float>();
  return true;
}

// a dense matrix like x, or nothing
bool like(PyObject *o, const at::Tensor &x, const void **p) {
  *p = nullptr;
  if (o == Py_None) return true;
  const at::Tensor *t = plain(o);
  if (!t || t->scalar_type() != x.scalar_type() || t->device() != x.device() || !t->is_contiguous() || t->sizes() != x.sizes()) return false;
  *p = t->data_ptr();
  return true;
}

const at::Tensor *rows_of(PyObject *o) {
  const at::Tensor *x = plain(o);
  return x && x->dim() == 2 && x->is_contiguous() && x->numel() > 0 && (x->scalar_type() == at::kHalf || x->scalar_type() == at::kFloat) ? x : nullptr;
}

PyObject *three(at::Tensor a, at::Tensor b, at::Tensor c) {
  PyObject *t = PyTuple_New(3);
  if (!t) return nullptr;
  PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(std::move(a)));
  PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(std::move(b)));
  PyTuple_SET_ITEM(t, 2, THPVariable_Wrap(std::move(c)));
  return t;
}

// bn_forward(x, residual, weight, bias, running mean, running variance, batch statistics, momentum, eps, act, slope, stream, batch count)
//   -> (y, mean, rstd), None or an error code
PyObject *bn_forward(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 13) {
    PyErr_SetString(PyExc_TypeError, "bn_forward: thirteen arguments");
    return nullptr;
  }
  const at::Tensor *x = rows_of(args[0]);
  if (!x) Py_RETURN_NONE;
  const int64_t n = x->size(0), c = x->size(1);
  const void *res;
  const float *w, *b, *mean, *var;
  if (!like(args[1], *x, &res) || !floats(args[2], x->device(), c, &w) || !floats(args[3], x->device(), c, &b) ||
      !floats(args[4], x->device(), c, &mean) || !floats(args[5], x->device(), c, &var))
    Py_RETURN_NONE;
  int64_t *batches = nullptr;
  if (args[12] != Py_None) {
    const at::Tensor *t = plain(args[12]);
    if (!t || t->scalar_type() != at::kLong || t->device() != x->device() || t->numel() != 1 || !pce_bn_forward_counted) Py_RETURN_NONE;
    batches = t->data_ptr<int64_t>();
  }
  const int batch = PyObject_IsTrue(args[6]), act = (int)PyLong_AsLong(args[9]), dt = x->scalar_type() == at::kHalf ? PCE_F16 : PCE_F32;
  const float momentum = (float)PyFloat_AsDouble(args[7]), eps = (float)PyFloat_AsDouble(args[8]), slope = (float)PyFloat_AsDouble(args[10]);
  void *stream = PyLong_AsVoidPtr(args[11]);
  if (PyErr_Occurred()) return nullptr;
  at::Tensor y, save, ws;
  int rc;
  {
    Unlocked unlocked;
    const int64_t ws_bytes = pce_bn_workspace_bytes(n, (int32_t)c);
    y = at::empty({n, c}, x->options());
    save = at::empty({2 * c}, x->options().dtype(at::kFloat));
    ws = at::empty({ws_bytes}, x->options().dtype(at::kByte));
    float *s = save.data_ptr<float>();
    float *m = const_cast<float *>(mean), *v = const_cast<float *>(var);
    rc = batches ? pce_bn_forward_counted(x->data_ptr(), res, y.data_ptr(), dt, n, (int32_t)c, w, b, m, v, batches, batch, momentum, eps, s, s + c,
                                          ws.data_ptr(), ws_bytes, act, slope, stream)
                 : pce_bn_forward(x->data_ptr(), res, y.data_ptr(), dt, n, (int32_t)c, w, b, m, v, batch, momentum, eps, s, s + c, ws.data_ptr(),
                                  ws_bytes, act, slope, stream);
  }
  if (rc != PCE_OK) return PyLong_FromLong(rc);
  return three(std::move(y), part(save, 0, c), part(save, c, c));
  END_HANDLE_TH_ERRORS
}

// bn_backward(x, dy, y, weight, mean, rstd, batch statistics, act, slope, stream, masked)
//   -> (dx, grad of weight, grad of bias[, masked dy]), None or an error code
PyObject *bn_backward(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 11) {
    PyErr_SetString(PyExc_TypeError, "bn_backward: eleven arguments");
    return nullptr;
  }
  const at::Tensor *x = rows_of(args[0]);
  if (!x) Py_RETURN_NONE;
  const int64_t n = x->size(0), c = x->size(1);
  const void *dy, *y;
  const float *w, *mean, *rstd;
  if (!like(args[1], *x, &dy) || !dy || !like(args[2], *x, &y) || !floats(args[3], x->device(), c, &w) || !floats(args[4], x->device(), c, &mean) ||
      !floats(args[5], x->device(), c, &rstd) || !mean || !rstd)
    Py_RETURN_NONE;
  const int batch = PyObject_IsTrue(args[6]), act = (int)PyLong_AsLong(args[7]), dt = x->scalar_type() == at::kHalf ? PCE_F16 : PCE_F32;
  const float slope = (float)PyFloat_AsDouble(args[8]);
  void *stream = PyLong_AsVoidPtr(args[9]);
  const int mask = PyObject_IsTrue(args[10]);
  if (PyErr_Occurred()) return nullptr;
  if (mask && (act == PCE_ACT_NONE || !pce_bn_backward_masked)) Py_RETURN_NONE;
  if (act != PCE_ACT_NONE && (!y || (act == PCE_ACT_LEAKY_RELU && !(slope > 0)))) Py_RETURN_NONE;
  at::Tensor dx, grads, ws, masked;
  int rc;
  {
    Unlocked unlocked;
    const int64_t ws_bytes = pce_bn_workspace_bytes(n, (int32_t)c);
    dx = at::empty({n, c}, x->options());
    grads = at::empty({2 * c}, x->options().dtype(at::kFloat));
    ws = at::empty({ws_bytes}, x->options().dtype(at::kByte));
    float *g = grads.data_ptr<float>();
    if (mask) masked = at::empty({n, c}, x->options());
    const void *out = act == PCE_ACT_NONE ? nullptr : y;
    rc = mask ? pce_bn_backward_masked(x->data_ptr(), dy, out, act, slope, masked.data_ptr(), dx.data_ptr(), dt, n, (int32_t)c, w, mean, rstd, batch,
                                       g, g + c, ws.data_ptr(), ws_bytes, stream)
              : pce_bn_backward(x->data_ptr(), dy, out, act, slope, dx.data_ptr(), dt, n, (int32_t)c, w, mean, rstd, batch, g, g + c, ws.data_ptr(),
                                ws_bytes, stream);
  }
  if (rc != PCE_OK) return PyLong_FromLong(rc);
  PyObject *t = three(std::move(dx), part(grads, 0, c), part(grads, c, c));
  if (t && mask && _PyTuple_Resize(&t, 4) == 0) PyTuple_SET_ITEM(t, 3, THPVariable_Wrap(std::move(masked)));
  return t;
  END_HANDLE_TH_ERRORS
}

// wgrad(features, output gradient, imap, omap, kpos, qkpos, n_in, n_out, kv, mid, qsum, stream[, zeros to add to])
//   -> fp32 [kv, c_in, c_out], None or an error code
PyObject *wgrad(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 12 && n_args != 13) {
    PyErr_SetString(PyExc_TypeError, "wgrad: twelve or thirteen arguments");
    return nullptr;
  }
  const at::Tensor *x = rows_of(args[0]), *g = rows_of(args[1]);
  if (!x || !g || x->scalar_type() != g->scalar_type() || x->device() != g->device()) Py_RETURN_NONE;
  int64_t num[5];
  for (int i = 0; i < 5; ++i) num[i] = PyLong_AsLongLong(args[6 + i]);
  void *stream = PyLong_AsVoidPtr(args[11]);
  if (PyErr_Occurred()) return nullptr;
  if (x->size(0) != num[0] || g->size(0) != num[1]) Py_RETURN_NONE;
  PyObject *tuple = PyTuple_Pack(4, args[2], args[3], args[4], args[5]);
  if (!tuple) return nullptr;
  View v{tuple};
  const int32_t *m[4];
  for (int i = 0; i < 4; ++i) m[i] = v.array(i, x->device());
  Py_DECREF(tuple);   // (the caller holds the tensors)
  if (v.bad || num[2] <= 0) Py_RETURN_NONE;
  const int64_t c_in = x->size(1), c_out = g->size(1);
  const at::Tensor *zeros = nullptr;
  if (n_args == 13 && args[12] != Py_None) {
    zeros = plain(args[12]);
    if (!zeros || zeros->scalar_type() != at::kFloat || zeros->device() != x->device() || !zeros->is_contiguous() ||
        zeros->numel() != num[2] * c_in * c_out || !pce_conv_wgrad_add)
      Py_RETURN_NONE;
  }
  at::Tensor gw;
  int rc;
  {
    Unlocked unlocked;
    if (!zeros) gw = at::empty({num[2], c_in, c_out}, x->options().dtype(at::kFloat));
    float *to = zeros ? zeros->data_ptr<float>() : gw.data_ptr<float>();
    const int dt = x->scalar_type() == at::kHalf ? PCE_F16 : PCE_F32, ci = (int)c_in, co = (int)c_out, kv = (int)num[2], mid = (int)num[3];
    rc = zeros ? pce_conv_wgrad_add(x->data_ptr(), g->data_ptr(), dt, num[0], num[1], ci, co, kv, mid, m[0], m[1], m[2], m[3], num[4], to, stream)
               : pce_conv_wgrad(x->data_ptr(), g->data_ptr(), dt, num[0], num[1], ci, co, kv, mid, m[0], m[1], m[2], m[3], num[4], to, stream);
  }
  if (rc != PCE_OK) return PyLong_FromLong(rc);
  if (!zeros) return THPVariable_Wrap(std::move(gw));
  Py_INCREF(args[12]);
  return args[12];
  END_HANDLE_TH_ERRORS
}

// piece(bytes, offset, rows, columns, like): a [rows, columns] matrix of like's type in the memory of `bytes` from byte `offset`
PyObject *piece(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 5 || !THPVariable_Check(args[0]) || !THPVariable_Check(args[4])) {
    PyErr_SetString(PyExc_TypeError, "piece: two tensors around three numbers");
    return nullptr;
  }
  const at::Tensor &bytes = THPVariable_Unpack(args[0]), &like = THPVariable_Unpack(args[4]);
  const int64_t off = PyLong_AsLongLong(args[1]), rows = PyLong_AsLongLong(args[2]), cols = PyLong_AsLongLong(args[3]);
  if (PyErr_Occurred()) return nullptr;
  const int64_t size = (int64_t)like.element_size(), from = (int64_t)bytes.storage_offset() + off;
  if (bytes.scalar_type() != at::kByte || off < 0 || rows < 0 || cols < 0 || from % size || off + rows * cols * size > bytes.numel()) {
    PyErr_SetString(PyExc_ValueError, "piece: outside the buffer");
    return nullptr;
  }
  at::Tensor t = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(bytes.storage()), c10::DispatchKeySet(c10::DispatchKey::CUDA), like.dtype());
  t.unsafeGetTensorImpl()->set_storage_offset(from / size);
  t.unsafeGetTensorImpl()->set_sizes_contiguous({rows, cols});
  return THPVariable_Wrap(std::move(t));
  END_HANDLE_TH_ERRORS
}

// cut(array, first, count) -> elements `first` .. of a vector of int32, in its memory; None where the caller has to slice it
PyObject *cut(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 3) {
    PyErr_SetString(PyExc_TypeError, "cut: a tensor and two numbers");
    return nullptr;
  }
  const at::Tensor *t = plain(args[0]);
  const int64_t first = PyLong_AsLongLong(args[1]), count = PyLong_AsLongLong(args[2]);
  if (PyErr_Occurred()) return nullptr;
  if (!t || t->scalar_type() != at::kInt || t->dim() != 1 || !t->is_contiguous() || first < 0 || count < 0 || first > t->numel() - count) Py_RETURN_NONE;
  return THPVariable_Wrap(part(*t, first, count));
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {{"layer", (PyCFunction)(void (*)())layer, METH_FASTCALL, nullptr},
                         {"bn_forward", (PyCFunction)(void (*)())bn_forward, METH_FASTCALL, nullptr},
                         {"bn_backward", (PyCFunction)(void (*)())bn_backward, METH_FASTCALL, nullptr},
                         {"wgrad", (PyCFunction)(void (*)())wgrad, METH_FASTCALL, nullptr},
                         {"piece", (PyCFunction)(void (*)())piece, METH_FASTCALL, nullptr},
                         {"cut", (PyCFunction)(void (*)())cut, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "Host side of a forward layer", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// the torch and the Python this was compiled against; the front end looks for it before it loads the file (_lib.host_is_current)
extern "C" __attribute__((used, visibility("default"))) const char pce_host_stamp[] = PCE_HOST_STAMP;

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&module); }
