// The operator calls' common case without an interpreter in between: operands as the library takes them (exact
// torch.Tensors on the GPU, contiguous, of the right types and shapes; plain ints and tuples of them).  Each function
// checks that, allocates the result, calls the library and returns the tensor; for anything else, and for any error, it
// returns None, and the Python operator of the same name (ops.py) takes the call from the beginning, with its conversions and
// its messages.
//
// Why: a launch-sized operator is 3.5 - 4.5 us of GPU time, and checking, allocating and calling through ctypes from Python
// was 6.3 us of host time.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <climits>

#include "../../include/unit_amd.h"

namespace {

// the library's functions, by the addresses of the instance that ctypes loaded (bind)
struct Library {
  decltype(&unit_conv_out_hw) conv_out_hw;
  decltype(&unit_conv2d_nchwc_u8s8s32) conv_u8;
  decltype(&unit_conv2d_nchwc_u8s8s32_prepared) conv_u8_prepared;
  decltype(&unit_conv2d_nchwc_s8s8s32_fused) fused;
  decltype(&unit_conv2d_nchwc_s8s8s32_fused_prepared) fused_prepared;
  decltype(&unit_conv2d_nchwc_u8s8u8_requant_prepared) requant;
  decltype(&unit_conv3d_ncdhwc_s8s8s32) conv3d;
  decltype(&unit_conv2d_nchw16c_f16f32) conv_f16;
  decltype(&unit_conv2d_nchw16c_f16f32_prepared) conv_f16_prepared;
  decltype(&unit_conv2d_nchw_f16f32) conv_f16_plain;
  decltype(&unit_conv2d_nchw_f16f32_ws_bytes) conv_f16_plain_bytes;
  decltype(&unit_dense_dotprod_u8s8s32) dense_packed;
  decltype(&unit_dense_u8s8s32) dense;
  decltype(&unit_dense_u8s8s32_prepared) dense_prepared;
  decltype(&unit_gemm_f16) gemm;
  decltype(&unit_gemm_f16_prepared) gemm_prepared;
  decltype(&unit_gemm_f16_ws) gemm_ws;
};
Library lib;
constexpr int kFunctions = sizeof(Library) / sizeof(void *);

// ops.PreparedConvWeight, PreparedDenseWeight, PreparedGemmB; torch.int8, torch.float16
PyObject *conv_weight_type, *dense_weight_type, *gemm_b_type, *dtype_s8, *dtype_f16;
PyObject *n_buf, *n_K, *n_C, *n_KH, *n_KW, *n_cb, *n_dtype, *n_w, *n_wsum, *n_bt, *n_N;

// a tensor the library can be handed as it is, or null
const at::Tensor *operand(PyObject *o, at::ScalarType type, int dim) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor &t = THPVariable_Unpack(o);
  // has_storage: the wrapped tensors of torch.func's transforms are torch.Tensors too, and have no data pointer
  return t.is_cuda() && t.has_storage() && t.scalar_type() == type && t.dim() == dim && t.layout() == at::kStrided && t.is_contiguous()
             ? &t
             : nullptr;
}

bool number(PyObject *o, int32_t *v) {
  if (!PyLong_CheckExact(o)) return false;
  int over = 0;
  const long x = PyLong_AsLongAndOverflow(o, &over);
  if (over || x < INT_MIN || x > INT_MAX) return false;
  *v = (int32_t)x;
  return true;
}

bool pair(PyObject *o, int32_t *a, int32_t *b) {
  if (PyTuple_CheckExact(o))
    return PyTuple_GET_SIZE(o) == 2 && number(PyTuple_GET_ITEM(o, 0), a) && number(PyTuple_GET_ITEM(o, 1), b);
  if (!number(o, a)) return false;
  *b = *a;
  return true;
}

bool padding(PyObject *o, unit_conv_desc *d) {  // as ops._pad4
  if (PyTuple_CheckExact(o)) {
    if (PyTuple_GET_SIZE(o) == 4)
      return number(PyTuple_GET_ITEM(o, 0), &d->pt) && number(PyTuple_GET_ITEM(o, 1), &d->pl) &&
             number(PyTuple_GET_ITEM(o, 2), &d->pb) && number(PyTuple_GET_ITEM(o, 3), &d->pr);
    if (!pair(o, &d->pt, &d->pl)) return false;
    d->pb = d->pt, d->pr = d->pl;
    return true;
  }
  if (!number(o, &d->pt)) return false;
  d->pl = d->pb = d->pr = d->pt;
  return true;
}

bool attribute(PyObject *o, PyObject *name, int32_t *v) {
  PyObject *a = PyObject_GetAttr(o, name);
  if (!a) return PyErr_Clear(), false;
  const bool ok = number(a, v);
  Py_DECREF(a);
  return ok;
}

// an attribute that is a tensor on `like`'s device
bool attribute(PyObject *o, PyObject *name, at::ScalarType type, int dim, const at::Tensor &like, at::Tensor *t) {
  PyObject *a = PyObject_GetAttr(o, name);
  if (!a) return PyErr_Clear(), false;
  const at::Tensor *p = operand(a, type, dim);
  const bool ok = p && p->device() == like.device();
  if (ok) *t = *p;
  Py_DECREF(a);
  return ok;
}

// a PreparedConvWeight: window and channels into the descriptor
bool prepared_conv(PyObject *o, PyObject *dtype, const at::Tensor &data, unit_conv_desc *d, at::Tensor *buf) {
  int32_t c, cb;
  PyObject *t = PyObject_GetAttr(o, n_dtype);
  if (!t) return PyErr_Clear(), false;
  Py_DECREF(t);
  return t == dtype && attribute(o, n_buf, at::kByte, 1, data, buf) && attribute(o, n_K, &d->K) && attribute(o, n_C, &c) &&
         attribute(o, n_KH, &d->KH) && attribute(o, n_KW, &d->KW) && attribute(o, n_cb, &cb) && c == d->C && cb == d->cb;
}

bool small(const at::Tensor &t) {  // sizes that fit a descriptor's fields
  for (const int64_t s : t.sizes())
    if (s > INT_MAX) return false;
  return true;
}

void *stream() { return c10::hip::getCurrentHIPStream().stream(); }

at::Tensor result(const at::Tensor &like, at::IntArrayRef shape, at::ScalarType type) {
  return at::empty(shape, like.options().dtype(type));
}

// other Python threads run while one is in scope, also out of which an exception leads
struct WithoutGil {
  PyThreadState *state = PyEval_SaveThread();
  ~WithoutGil() { PyEval_RestoreThread(state); }
};

// call(stream, operands..., result), with data pointers for the tensors (taken first: that may throw)
template <class F, class... T>
PyObject *finish(at::Tensor &&out, F &&call, const T &...operands) {
  int rc;
  const auto run = [&](auto... p) {
    void *const s = stream(), *const o = out.data_ptr();
    WithoutGil others;
    rc = call(s, p..., o);
  };
  run(operands.data_ptr()...);
  if (rc != UNIT_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
}

// no C++ exception leaves a function: the Python operator meets the same condition again and reports it
template <PyObject *(*F)(PyObject *const *, Py_ssize_t)>
PyObject *guarded(PyObject *, PyObject *const *args, Py_ssize_t n) {
  try {
    return F(args, n);
  } catch (...) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
}

// data and window of a blocked 2-D convolution: descriptor, and the weight's pointer (kept alive by the caller's object)
bool conv_operands(PyObject *data_o, PyObject *kernel_o, at::ScalarType type, unit_conv_desc *d, const at::Tensor **data,
                   at::Tensor *weight, bool *prepared) {
  const at::Tensor *x = operand(data_o, type, 5);
  if (!x || !small(*x)) return false;
  const bool half = type == at::kHalf;
  const int64_t cc = x->size(1), cb = x->size(4);
  if (cb != 16 && (half || cb != 4)) return false;
  if (cc * cb > INT_MAX) return false;
  d->N = (int32_t)x->size(0), d->C = (int32_t)(cc * cb), d->H = (int32_t)x->size(2), d->W = (int32_t)x->size(3), d->cb = (int32_t)cb;
  *data = x;
  *prepared = (PyObject *)Py_TYPE(kernel_o) == conv_weight_type;
  if (*prepared) return prepared_conv(kernel_o, half ? dtype_f16 : dtype_s8, *x, d, weight);
  const at::Tensor *w = half ? operand(kernel_o, at::kHalf, 6) : operand(kernel_o, at::kChar, 7);
  if (!w || !small(*w) || w->size(0) > INT_MAX / 16 || w->size(1) != cc) return false;
  if (half ? (w->size(4) != 16 || w->size(5) != 16) : (w->size(4) != cb / 4 || w->size(5) != 16 || w->size(6) != 4)) return false;
  d->K = (int32_t)w->size(0) * 16, d->KH = (int32_t)w->size(2), d->KW = (int32_t)w->size(3);
  *weight = *w;
  return true;
}

bool out_hw(const unit_conv_desc &d, int32_t *oh, int32_t *ow) { return lib.conv_out_hw(&d, oh, ow) == UNIT_OK; }

// bias: None, or int32 of K values on the data's device
bool bias_of(PyObject *o, int32_t k, const at::Tensor &data, const int32_t **p) {
  *p = nullptr;
  if (o == Py_None) return true;
  if (!THPVariable_CheckExact(o)) return false;
  const at::Tensor &b = THPVariable_Unpack(o);
  if (b.scalar_type() != at::kInt || b.numel() != k || b.device() != data.device() || b.layout() != at::kStrided || !b.has_storage() ||
      !b.is_contiguous())
    return false;
  *p = static_cast<const int32_t *>(b.data_ptr());
  return true;
}

// (data, kernel, stride, padding, dilation)
PyObject *conv_u8(PyObject *const *a, Py_ssize_t n) {
  unit_conv_desc d;
  const at::Tensor *x;
  at::Tensor w;
  bool prepared;
  int32_t oh, ow;
  if (n != 5 || !conv_operands(a[0], a[1], at::kByte, &d, &x, &w, &prepared) || !pair(a[2], &d.sh, &d.sw) || !padding(a[3], &d) ||
      !pair(a[4], &d.dh, &d.dw) || !out_hw(d, &oh, &ow))
    Py_RETURN_NONE;
  at::Tensor out = result(*x, {d.N, d.K / 16, oh, ow, 16}, at::kInt);
  return finish(std::move(out), [&](void *s, void *xp, void *wp, void *o) {
    return (prepared ? lib.conv_u8_prepared : lib.conv_u8)(&d, xp, wp, o, s);
  }, *x, w);
}

// (data, kernel, bias, scale, stride, padding, dilation)
PyObject *conv_fused(PyObject *const *a, Py_ssize_t n) {
  unit_conv_desc d;
  const at::Tensor *x;
  at::Tensor w;
  bool prepared;
  const int32_t *bias;
  int32_t oh, ow, scale;
  if (n != 7 || !conv_operands(a[0], a[1], at::kChar, &d, &x, &w, &prepared) || !bias_of(a[2], d.K, *x, &bias) || !number(a[3], &scale) ||
      !pair(a[4], &d.sh, &d.sw) || !padding(a[5], &d) || !pair(a[6], &d.dh, &d.dw) || !out_hw(d, &oh, &ow))
    Py_RETURN_NONE;
  at::Tensor out = result(*x, {d.N, d.K / 16, oh, ow, 16}, at::kInt);
  return finish(std::move(out), [&](void *s, void *xp, void *wp, void *o) {
    return (prepared ? lib.fused_prepared : lib.fused)(&d, xp, wp, bias, scale, o, s);
  }, *x, w);
}

// (data, prepared kernel, bias, scale, shift, stride, padding, dilation)
PyObject *conv_requant(PyObject *const *a, Py_ssize_t n) {
  unit_conv_desc d;
  const at::Tensor *x;
  at::Tensor w;
  bool prepared;
  const int32_t *bias;
  int32_t oh, ow, scale, shift;
  if (n != 8 || !conv_operands(a[0], a[1], at::kByte, &d, &x, &w, &prepared) || !prepared || !bias_of(a[2], d.K, *x, &bias) ||
      !number(a[3], &scale) || !number(a[4], &shift) || !pair(a[5], &d.sh, &d.sw) || !padding(a[6], &d) || !pair(a[7], &d.dh, &d.dw) ||
      !out_hw(d, &oh, &ow))
    Py_RETURN_NONE;
  at::Tensor out = result(*x, {d.N, d.K / 16, oh, ow, 16}, at::kByte);
  return finish(std::move(out), [&](void *s, void *xp, void *wp, void *o) { return lib.requant(&d, xp, wp, bias, scale, shift, o, s); }, *x,
                w);
}

// (data, kernel, stride)
PyObject *conv3d(PyObject *const *a, Py_ssize_t n) {
  if (n != 3) Py_RETURN_NONE;
  const at::Tensor *x = operand(a[0], at::kChar, 6), *w = operand(a[1], at::kChar, 8);
  unit_conv3d_desc d;
  if (!x || !w || !small(*x) || !small(*w) || !number(a[2], &d.stride) || d.stride <= 0) Py_RETURN_NONE;
  const int64_t cc = x->size(1), cb = x->size(5);
  if ((cb != 16 && cb != 4) || cc * cb > INT_MAX || (cb == 4 && (cc * cb) % 16 == 0) || w->size(0) > INT_MAX / 16) Py_RETURN_NONE;
  if (w->size(1) != cc || w->size(5) != cb / 4 || w->size(6) != 16 || w->size(7) != 4) Py_RETURN_NONE;
  d.N = (int32_t)x->size(0), d.C = (int32_t)(cc * cb), d.D = (int32_t)x->size(2), d.H = (int32_t)x->size(3), d.W = (int32_t)x->size(4);
  d.K = (int32_t)w->size(0) * 16, d.KD = (int32_t)w->size(2), d.KH = (int32_t)w->size(3), d.KW = (int32_t)w->size(4);
  if (d.KD > d.D || d.KH > d.H || d.KW > d.W) Py_RETURN_NONE;
  at::Tensor out = result(*x, {d.N, d.K / 16, (d.D - d.KD) / d.stride + 1, (d.H - d.KH) / d.stride + 1, (d.W - d.KW) / d.stride + 1, 16},
                          at::kInt);
  return finish(std::move(out), [&](void *s, void *xp, void *wp, void *o) { return lib.conv3d(&d, xp, wp, o, s); }, *x, *w);
}

// (a, b, stride_h, stride_w): blocked a with blocked or prepared b, or both plain
PyObject *conv_f16(PyObject *const *a, Py_ssize_t n) {
  unit_conv_desc d{};
  int32_t oh, ow;
  if (n != 4 || !number(a[2], &d.sh) || !number(a[3], &d.sw)) Py_RETURN_NONE;
  d.dh = d.dw = 1;
  const at::Tensor *x = operand(a[0], at::kHalf, 4);
  if (x) {
    const at::Tensor *w = operand(a[1], at::kHalf, 4);
    if (!w || !small(*x) || !small(*w) || w->size(1) != x->size(1) || x->size(1) % 16 || w->size(0) % 16) Py_RETURN_NONE;
    d.N = (int32_t)x->size(0), d.C = (int32_t)x->size(1), d.H = (int32_t)x->size(2), d.W = (int32_t)x->size(3), d.cb = 16;
    d.K = (int32_t)w->size(0), d.KH = (int32_t)w->size(2), d.KW = (int32_t)w->size(3);
    // the prepared form fills 32-channel blocks; past the size limit the operator packs the operands instead
    if ((double)((d.K + 31) / 32) * 64 * d.C * d.KH * d.KW > 2147483647.0 || !out_hw(d, &oh, &ow)) Py_RETURN_NONE;
    size_t need = 0;
    if (lib.conv_f16_plain_bytes(&d, &need) != UNIT_OK || need == 0) Py_RETURN_NONE;
    at::Tensor ws = result(*x, {(int64_t)need}, at::kByte), out = result(*x, {d.N, d.K / 16, oh, ow, 16}, at::kFloat);
    return finish(std::move(out), [&](void *s, void *xp, void *wp, void *sp, void *o) { return lib.conv_f16_plain(&d, xp, wp, o, sp, need, s); },
                  *x, *w, ws);
  }
  at::Tensor w;
  bool prepared;
  if (!conv_operands(a[0], a[1], at::kHalf, &d, &x, &w, &prepared) || !out_hw(d, &oh, &ow)) Py_RETURN_NONE;
  at::Tensor out = result(*x, {d.N, d.K / 16, oh, ow, 16}, at::kFloat);
  return finish(std::move(out), [&](void *s, void *xp, void *wp, void *o) {
    return (prepared ? lib.conv_f16_prepared : lib.conv_f16)(&d, xp, wp, o, s);
  }, *x, w);
}

// (data, weight): packed, row-major or prepared
PyObject *dense(PyObject *const *a, Py_ssize_t n) {
  if (n != 2) Py_RETURN_NONE;
  const at::Tensor *x = operand(a[0], at::kByte, 2);
  if (!x || !small(*x)) Py_RETURN_NONE;
  const int32_t m = (int32_t)x->size(0), k = (int32_t)x->size(1);
  if ((PyObject *)Py_TYPE(a[1]) == dense_weight_type) {
    at::Tensor w, sums;
    if (!attribute(a[1], n_w, at::kChar, 2, *x, &w) || !attribute(a[1], n_wsum, at::kInt, 1, *x, &sums) || !small(w) || w.size(1) != k ||
        sums.size(0) != w.size(0))
      Py_RETURN_NONE;
    const int32_t nn = (int32_t)w.size(0);
    at::Tensor out = result(*x, {m, nn}, at::kInt);
    return finish(std::move(out), [&](void *s, void *xp, void *wp, void *sp, void *o) {
      return lib.dense_prepared(xp, wp, static_cast<int *>(sp), o, m, nn, k, s);
    }, *x, w, sums);
  }
  if (const at::Tensor *w = operand(a[1], at::kChar, 4)) {
    if (w->size(2) != 128 || w->size(3) != 4 || w->size(1) * 4 != k || w->size(0) > INT_MAX / 128) Py_RETURN_NONE;
    const int32_t nn = (int32_t)w->size(0) * 128;
    at::Tensor out = result(*x, {m, nn}, at::kInt);
    return finish(std::move(out), [&](void *s, void *xp, void *wp, void *o) { return lib.dense_packed(xp, wp, o, m, nn, k, s); }, *x, *w);
  }
  const at::Tensor *w = operand(a[1], at::kChar, 2);
  if (!w || !small(*w) || w->size(1) != k) Py_RETURN_NONE;
  const int32_t nn = (int32_t)w->size(0);
  at::Tensor out = result(*x, {m, nn}, at::kInt);
  return finish(std::move(out), [&](void *s, void *xp, void *wp, void *o) { return lib.dense(xp, wp, o, m, nn, k, s); }, *x, *w);
}

// (a, b, fp16 result?, workspace or None): b (K, N) or prepared
PyObject *gemm(PyObject *const *a, Py_ssize_t n) {
  if (n != 4) Py_RETURN_NONE;
  const at::Tensor *x = operand(a[0], at::kHalf, 2);
  if (!x || !small(*x)) Py_RETURN_NONE;
  const int32_t m = (int32_t)x->size(0), k = (int32_t)x->size(1), half = a[2] == Py_True;
  const at::ScalarType type = half ? at::kHalf : at::kFloat;
  if ((PyObject *)Py_TYPE(a[1]) == gemm_b_type) {
    at::Tensor bt;
    int32_t kk, nn;
    if (!attribute(a[1], n_bt, at::kHalf, 2, *x, &bt) || !attribute(a[1], n_K, &kk) || !attribute(a[1], n_N, &nn) || kk != k ||
        bt.size(0) != nn || bt.size(1) != k)
      Py_RETURN_NONE;
    at::Tensor out = result(*x, {m, nn}, type);
    return finish(std::move(out), [&](void *s, void *xp, void *bp, void *o) { return lib.gemm_prepared(xp, bp, o, m, nn, k, half, s); }, *x, bt);
  }
  const at::Tensor *b = operand(a[1], at::kHalf, 2);
  if (!b || !small(*b) || b->size(0) != k) Py_RETURN_NONE;
  const int32_t nn = (int32_t)b->size(1);
  if (a[3] != Py_None) {
    if (!THPVariable_CheckExact(a[3])) Py_RETURN_NONE;
    const at::Tensor &ws = THPVariable_Unpack(a[3]);
    if (!ws.is_cuda() || !ws.has_storage() || ws.scalar_type() != at::kByte || ws.layout() != at::kStrided || !ws.is_contiguous())
      Py_RETURN_NONE;
    at::Tensor out = result(*x, {m, nn}, type);
    const size_t bytes = (size_t)ws.numel();
    return finish(std::move(out), [&](void *s, void *xp, void *bp, void *sp, void *o) {
      return lib.gemm_ws(xp, bp, o, m, nn, k, half, sp, bytes, s);
    }, *x, *b, ws);
  }
  at::Tensor out = result(*x, {m, nn}, type);
  return finish(std::move(out), [&](void *s, void *xp, void *bp, void *o) { return lib.gemm(xp, bp, o, m, nn, k, half, s); }, *x, *b);
}

// (addresses in Library's order, the three prepared classes, torch.int8, torch.float16)
PyObject *bind(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (n != 6 || !PyTuple_CheckExact(a[0]) || PyTuple_GET_SIZE(a[0]) != kFunctions) {
    PyErr_SetString(PyExc_ValueError, "bind: unexpected arguments");
    return nullptr;
  }
  void *f[kFunctions];
  for (int i = 0; i < kFunctions; ++i) {
    f[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(a[0], i));
    if (!f[i]) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: null address");
      return nullptr;
    }
  }
  memcpy(&lib, f, sizeof lib);
  PyObject **const kept[] = {&conv_weight_type, &dense_weight_type, &gemm_b_type, &dtype_s8, &dtype_f16};
  for (int i = 0; i < 5; ++i) {
    Py_INCREF(a[i + 1]);
    Py_XDECREF(*kept[i]);
    *kept[i] = a[i + 1];
  }
  Py_RETURN_NONE;
}

template <PyObject *(*F)(PyObject *const *, Py_ssize_t)>
constexpr PyMethodDef method(const char *name) {
  return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(guarded<F>)), METH_FASTCALL, nullptr};
}

PyMethodDef methods[] = {
    method<conv_u8>("conv_u8"),   method<conv_fused>("conv_fused"), method<conv_requant>("conv_requant"), method<conv3d>("conv3d"),
    method<conv_f16>("conv_f16"), method<dense>("dense"),           method<gemm>("gemm"),
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(bind)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject *PyInit__calls() {
  struct {
    PyObject **name;
    const char *text;
  } const names[] = {{&n_buf, "buf"}, {&n_K, "K"},         {&n_C, "C"}, {&n_KH, "KH"},     {&n_KW, "KW"}, {&n_cb, "cb"},
                     {&n_N, "N"},     {&n_dtype, "dtype"}, {&n_w, "w"}, {&n_wsum, "wsum"}, {&n_bt, "bt"}};
  for (const auto &x : names)
    if (!(*x.name = PyUnicode_InternFromString(x.text))) return nullptr;
  return PyModule_Create(&module);
}
