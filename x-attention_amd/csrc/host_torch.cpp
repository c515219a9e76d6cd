// Native host path of the Python package: reads sizes, strides and pointers straight from the tensors, allocates the
// output and one workspace from torch's caching allocator, and enqueues through the C ABI of libxattn_hip.so on the
// current stream.
//
// The short calls - a prompt of a thousand tokens, a decode step - are bound by host time when every size is a Python
// attribute lookup and every launch a ctypes call with forty conversions.  Each function here handles the ordinary
// form of its call and returns None for anything else (tensors to be made contiguous, other devices, arguments to be
// refused); the Python code then takes over, and raises where there is something to raise.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <optional>

#include "xattn_hip.h"

namespace {

// A bf16 tensor on a ROCm device as the kernels read it: feature dimension contiguous, 16-byte aligned rows.
inline bool kernel_ready(const at::Tensor& t, int64_t dim) {
  const int64_t n = t.dim();
  return t.is_cuda() && t.scalar_type() == at::kBFloat16 && n == dim && t.size(n - 1) == 128 && t.stride(n - 1) == 1 &&
         t.stride(n - 2) % 8 == 0 && t.stride(n - 3) % 8 == 0 && (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
}

inline const at::Tensor* tensor_of(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

// Makes a tensor's device current for the launches, and only if it is not.
struct OnDevice {
  explicit OnDevice(c10::Device d) {
    if (c10::hip::current_device() != d.index()) guard.emplace(d);
  }
  std::optional<c10::DeviceGuard> guard;
};

inline void* stream_of(c10::Device d) { return static_cast<void*>(c10::hip::getCurrentHIPStream(d.index()).stream()); }

PyObject* fail(const char* what, int code) {
  // the package's own error type, looked up only when something went wrong
  PyObject* mod = PyImport_ImportModule("xattn.src.hip_backend");
  PyObject* type = mod ? PyObject_GetAttrString(mod, "XattnHipError") : nullptr;
  if (type) PyErr_Format(type, "%s failed: %s (code %d)", what, xattn_error_string(code), code);
  Py_XDECREF(type);
  Py_XDECREF(mod);
  return nullptr;
}

// Thresholds of a call: host values (one, or one per head), or a float64 [H] device tensor.
struct Tau {
  double host[64];
  int count = 0;
  at::Tensor device;
};

bool read_tau(PyObject* o, int64_t heads, c10::Device dev, Tau* tau) {
  const at::Tensor* t = tensor_of(o);
  if (!t) {
    tau->host[0] = PyFloat_AsDouble(o);
    if (PyErr_Occurred()) {
      PyErr_Clear();
      return false;
    }
    tau->count = 1;
    return true;
  }
  const int64_t n = t->numel();
  if (n != 1 && n != heads) return false;
  if (t->is_cpu() && n <= 64) {
    // a tensor keeps its own precision (xattn/src/utils.py:91-92): converted to double value by value, no copy to the
    // device and no wait for it
    const at::Tensor d = t->scalar_type() == at::kDouble && t->is_contiguous() ? *t : t->detach().to(at::kDouble).contiguous();
    const double* src = d.const_data_ptr<double>();
    for (int64_t i = 0; i < n; ++i) tau->host[i] = src[i];
    tau->count = (int)n;
    return true;
  }
  tau->device = t->detach().to(at::kDouble).reshape({-1}).expand({heads}).contiguous().to(dev);
  return true;
}

// What prefill and estimate share: geometry of a call and which rows and keys the reference's branches hide (see _Plan in
// xattn/src/Xattention.py of this package).
struct Call {
  int64_t H, Hkv, Lq, Lk, chunk;
  int stride, causal, own_chunk, zero_from;
  float scale;
  // false: not an ordinary call
  bool read(const at::Tensor& q, const at::Tensor& k, long stride_, double norm, int use_triton, int causal_, long chunk_) {
    if (!kernel_ready(q, 4) || !kernel_ready(k, 4) || k.device() != q.device()) return false;
    H = q.size(1), Lq = q.size(2), Hkv = k.size(1), Lk = k.size(2), chunk = chunk_;
    if (q.size(0) != 1 || k.size(0) != 1) return false;
    if ((stride_ != 4 && stride_ != 8 && stride_ != 16) || !(norm > 0) || H < 1 || Hkv < 1 || H % Hkv || Lq < 1 || Lk < Lq ||
        Lk > (int64_t(1) << 30) || chunk < 128 || chunk % 128 || chunk > (1 << 30))
      return false;
    if (padded(Lk) / 128 > 8192) return false;
    stride = (int)stride_;
    causal = causal_;
    const int64_t q_pad = padded(Lq) - Lq, k_pad = padded(Lk) - Lk, n_rq = padded(Lq) / stride;
    own_chunk = causal && !use_triton && k_pad / stride == 0;
    zero_from = (int)(use_triton ? std::max<int64_t>(0, n_rq - k_pad / stride) : n_rq - q_pad / stride);
    scale = (float)(1.0 / std::sqrt(128.0) / (double)stride / norm);
    return true;
  }
  int64_t padded(int64_t n) const { return (n + chunk - 1) / chunk * chunk; }
};

// prefill(q, k, v, stride, norm, threshold, use_triton, causal, chunk_size, keep_sink, keep_recent, workspace_limit)
PyObject* prefill(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 12) return PyErr_Format(PyExc_TypeError, "prefill takes 12 arguments");
  HANDLE_TH_ERRORS
  const at::Tensor *q = tensor_of(args[0]), *k = tensor_of(args[1]), *v = tensor_of(args[2]);
  if (!q || !k || !v) Py_RETURN_NONE;
  const long stride = PyLong_AsLong(args[3]);
  const double norm = PyFloat_AsDouble(args[4]);
  const long chunk = PyLong_AsLong(args[8]);
  const long long limit = PyLong_AsLongLong(args[11]);
  const int use_triton = PyObject_IsTrue(args[6]), causal = PyObject_IsTrue(args[7]);
  const int keep_sink = PyObject_IsTrue(args[9]), keep_recent = PyObject_IsTrue(args[10]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  Call c;
  if (!c.read(*q, *k, stride, norm, use_triton, causal, chunk) || !kernel_ready(*v, 4)) Py_RETURN_NONE;
  const c10::Device dev = q->device();
  if (v->device() != dev || v->size(0) != 1 || v->size(1) != c.Hkv || v->size(2) != c.Lk) Py_RETURN_NONE;
  const int H = (int)c.H, Lq = (int)c.Lq;
  size_t bytes = xattn_prefill_workspace_bytes(H, Lq, (int)c.Lk, c.stride, (int)chunk);
  if (bytes == 0 || (long long)bytes > limit) Py_RETURN_NONE;
  OnDevice on(dev);
  Tau tau;
  if (!read_tau(args[5], H, dev, &tau)) Py_RETURN_NONE;
  at::Tensor out = at::empty_strided({1, H, Lq, 128}, {(int64_t)Lq * H * 128, 128, (int64_t)H * 128, 1},
                                     at::TensorOptions().device(dev).dtype(at::kBFloat16));
  c10::DataPtr ws;
  try {
    ws = c10::hip::HIPCachingAllocator::get()->allocate(bytes);
  } catch (const c10::OutOfMemoryError&) {
    // most of it (up to 200 MB) is for lists cut into pieces: on a GPU that is full they stay whole
    const size_t least = xattn_prefill_least_workspace_bytes(H, Lq, (int)c.Lk, c.stride, (int)chunk);
    if (least >= bytes) throw;
    ws = c10::hip::HIPCachingAllocator::get()->allocate(bytes = least);
  }
  const int rc = xattn_prefill_fwd(
      q->data_ptr(), k->data_ptr(), v->data_ptr(), out.data_ptr(), ws.get(), bytes, H, (int)c.Hkv, Lq, (int)c.Lk, 128, q->stride(1),
      q->stride(2), k->stride(1), k->stride(2), v->stride(1), v->stride(2), 128, (int64_t)H * 128, c.stride, (int)chunk, causal,
      c.own_chunk, c.scale, c.zero_from, tau.count ? tau.host : nullptr, tau.count,
      tau.count ? nullptr : tau.device.const_data_ptr<double>(), keep_sink, keep_recent, (float)(1.0 / std::sqrt(128.0)), stream_of(dev));
  if (rc != XATTN_OK) return fail("xattn_prefill_fwd", rc);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// estimate(q, k, stride, norm, threshold, use_triton, causal, chunk_size, keep_sink, keep_recent, workspace_limit)
//   -> (block sums, mask) of xattn_estimate
PyObject* estimate(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 11) return PyErr_Format(PyExc_TypeError, "estimate takes 11 arguments");
  HANDLE_TH_ERRORS
  const at::Tensor *q = tensor_of(args[0]), *k = tensor_of(args[1]);
  if (!q || !k) Py_RETURN_NONE;
  const long stride = PyLong_AsLong(args[2]);
  const double norm = PyFloat_AsDouble(args[3]);
  const long chunk = PyLong_AsLong(args[7]);
  const long long limit = PyLong_AsLongLong(args[10]);
  const int use_triton = PyObject_IsTrue(args[5]), causal = PyObject_IsTrue(args[6]);
  const int keep_sink = PyObject_IsTrue(args[8]), keep_recent = PyObject_IsTrue(args[9]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  Call c;
  if (!c.read(*q, *k, stride, norm, use_triton, causal, chunk)) Py_RETURN_NONE;
  const c10::Device dev = q->device();
  const int H = (int)c.H, Lq = (int)c.Lq;
  const size_t bytes = xattn_estimate_workspace_bytes(H, Lq, (int)c.Lk, c.stride, 128, (int)chunk, 0);
  if (bytes == 0 || (long long)bytes > limit) Py_RETURN_NONE;
  OnDevice on(dev);
  Tau tau;
  if (!read_tau(args[4], H, dev, &tau)) Py_RETURN_NONE;
  const auto opts = at::TensorOptions().device(dev);
  at::Tensor sums = at::empty({1, H, c.padded(Lq) / 128, c.padded(c.Lk) / 128}, opts.dtype(at::kBFloat16));
  at::Tensor mask = at::empty(sums.sizes(), opts.dtype(at::kBool));
  const c10::DataPtr ws = c10::hip::HIPCachingAllocator::get()->allocate(bytes);
  const int rc = xattn_estimate_fwd(q->data_ptr(), k->data_ptr(), sums.data_ptr(), static_cast<uint8_t*>(mask.data_ptr()), ws.get(),
                                    bytes, H, (int)c.Hkv, Lq, (int)c.Lk, 128, q->stride(1), q->stride(2), k->stride(1), k->stride(2),
                                    c.stride, (int)chunk, causal, c.own_chunk, c.scale, c.zero_from, tau.count ? tau.host : nullptr,
                                    tau.count, tau.count ? nullptr : tau.device.const_data_ptr<double>(), keep_sink, keep_recent,
                                    stream_of(dev));
  if (rc != XATTN_OK) return fail("xattn_estimate_fwd", rc);
  PyObject* result = PyTuple_New(2);
  if (!result) return nullptr;
  PyTuple_SET_ITEM(result, 0, THPVariable_Wrap(std::move(sums)));
  PyTuple_SET_ITEM(result, 1, THPVariable_Wrap(std::move(mask)));
  return result;
  END_HANDLE_TH_ERRORS
}

// One decode step: heads of q, and heads and tokens of k and v, lie along the named dimensions; out is [H][128] in memory.
// None, and no error set: not an ordinary call.
PyObject* decode_step(const at::Tensor& q, int64_t q_head, const at::Tensor& k, const at::Tensor& v, int64_t head, int64_t token, double scale,
                      at::IntArrayRef out_sizes) {
  const int64_t H = q.size(q_head), Hkv = k.size(head), L = k.size(token);
  if (H < 1 || Hkv < 1 || H % Hkv || H / Hkv > 32 || L < 1 || L > (int64_t(1) << 30)) Py_RETURN_NONE;
  const size_t bytes = xattn_decode_workspace_bytes((int)H, (int)Hkv, (int)L);
  if (bytes == 0) Py_RETURN_NONE;
  const c10::Device dev = q.device();
  OnDevice on(dev);
  at::Tensor out = at::empty(out_sizes, at::TensorOptions().device(dev).dtype(at::kBFloat16));
  const c10::DataPtr ws = c10::hip::HIPCachingAllocator::get()->allocate(bytes);
  const int rc = xattn_decode_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), ws.get(), bytes, (int)H, (int)Hkv, (int)L, 128,
                                  q.stride(q_head), k.stride(head), k.stride(token), v.stride(head), v.stride(token), 128, (float)scale,
                                  stream_of(dev));
  if (rc != XATTN_OK) return fail("xattn_decode_fwd", rc);
  return THPVariable_Wrap(std::move(out));
}

// decode(q, k, v, token_major, sm_scale): single_decode_with_kv_cache without caller-provided buffers
PyObject* decode(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 5) return PyErr_Format(PyExc_TypeError, "decode takes 5 arguments");
  HANDLE_TH_ERRORS
  const at::Tensor *q = tensor_of(args[0]), *k = tensor_of(args[1]), *v = tensor_of(args[2]);
  if (!q || !k || !v) Py_RETURN_NONE;
  const int nhd = PyObject_IsTrue(args[3]);
  double scale = 1.0 / std::sqrt(128.0);
  if (args[4] != Py_None) scale = PyFloat_AsDouble(args[4]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  if (!q->is_cuda() || q->scalar_type() != at::kBFloat16 || q->dim() != 2 || q->size(1) != 128 || q->stride(1) != 1 ||
      q->stride(0) % 8 || (reinterpret_cast<uintptr_t>(q->data_ptr()) & 15))
    Py_RETURN_NONE;
  if (!kernel_ready(*k, 3) || !kernel_ready(*v, 3) || k->sizes() != v->sizes()) Py_RETURN_NONE;
  if (k->device() != q->device() || v->device() != q->device()) Py_RETURN_NONE;
  const int hd = nhd ? 1 : 0, td = 1 - hd;       // head and token dimension of k and v
  return decode_step(*q, 0, *k, *v, hd, td, scale, {q->size(0), 128});
  END_HANDLE_TH_ERRORS
}

// decode_layer(q, k, v): the decode step of an attention layer, q [1, heads, 1, 128] on k and v [1, kv_heads, tokens, 128], as its
// output projection takes it: [1, 1, heads * 128] (the views that decode() needs, and its result's, are 5 us of tensor calls)
PyObject* decode_layer(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 3) return PyErr_Format(PyExc_TypeError, "decode_layer takes 3 arguments");
  HANDLE_TH_ERRORS
  const at::Tensor *q = tensor_of(args[0]), *k = tensor_of(args[1]), *v = tensor_of(args[2]);
  if (!q || !k || !v || !kernel_ready(*q, 4) || !kernel_ready(*k, 4) || !kernel_ready(*v, 4)) Py_RETURN_NONE;
  if (q->size(0) != 1 || q->size(2) != 1 || k->size(0) != 1 || k->sizes() != v->sizes()) Py_RETURN_NONE;
  if (k->device() != q->device() || v->device() != q->device()) Py_RETURN_NONE;
  return decode_step(*q, 1, *k, *v, 1, 2, 1.0 / std::sqrt(128.0), {1, 1, q->size(1) * 128});
  END_HANDLE_TH_ERRORS
}

// A weight and bias (or None) as the projection kernels read them, on device dev.
struct Linear {
  const at::Tensor* w = nullptr;
  std::optional<at::Tensor> b;
  bool read(PyObject* weight, PyObject* bias, int64_t rows, int64_t width, c10::Device dev) {
    w = tensor_of(weight);
    if (!w || w->dim() != 2 || w->size(0) != rows || w->size(1) != width || w->stride(1) != 1 || w->stride(0) % 8 ||
        w->stride(0) < width || w->scalar_type() != at::kBFloat16 || w->device() != dev ||
        (reinterpret_cast<uintptr_t>(w->data_ptr()) & 15))
      return false;
    if (bias != Py_None) {
      const at::Tensor* t = tensor_of(bias);
      if (!t || t->dim() != 1 || t->size(0) != rows || t->stride(0) != 1 || t->scalar_type() != at::kBFloat16 || t->device() != dev)
        return false;
      b = *t;
    }
    return !at::GradMode::is_enabled() || (!w->requires_grad() && !(b && b->requires_grad()));
  }
  const void* bias_ptr() const { return b ? b->data_ptr() : nullptr; }
};

// Hidden states a layer's projections take natively: bf16 [1, tokens, width] without gaps, no autograd, no autocast.
const at::Tensor* hidden_of(PyObject* o) {
  const at::Tensor* x = tensor_of(o);
  if (!x || !x->is_cuda() || x->scalar_type() != at::kBFloat16 || x->dim() != 3 || x->size(0) != 1 || x->size(1) < 1 ||
      !x->is_contiguous() || x->size(2) % 8 || (reinterpret_cast<uintptr_t>(x->data_ptr()) & 15) ||
      (at::GradMode::is_enabled() && x->requires_grad()) || at::autocast::is_autocast_enabled(at::kCUDA))
    return nullptr;
  return x;
}

// project(hidden, wq, bq, wk, bk, wv, bv, cos, sin, heads, kv_heads) -> (q, k, v): the projections of a layer with q and
// k rotated, [1, heads, tokens, 128] views of token-major memory (what the projections write)
PyObject* project(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 11) return PyErr_Format(PyExc_TypeError, "project takes 11 arguments");
  HANDLE_TH_ERRORS
  const at::Tensor *x = hidden_of(args[0]), *cos = tensor_of(args[7]), *sin = tensor_of(args[8]);
  if (!x || !cos || !sin) Py_RETURN_NONE;
  const long heads[3] = {PyLong_AsLong(args[9]), PyLong_AsLong(args[10]), PyLong_AsLong(args[10])};
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const c10::Device dev = x->device();
  const int64_t L = x->size(1), K = x->size(2);
  if (heads[0] < 1 || heads[1] < 1 || heads[0] > 4096 || heads[1] > 4096 || L * (heads[0] + heads[1]) > 0x7fffffff) Py_RETURN_NONE;
  for (const at::Tensor* t : {cos, sin})
    if (t->dim() != 3 || t->size(0) != 1 || t->size(1) != L || t->size(2) != 128 || t->stride(2) != 1 || t->stride(1) % 8 ||
        t->scalar_type() != at::kBFloat16 || t->device() != dev || (reinterpret_cast<uintptr_t>(t->data_ptr()) & 15))
      Py_RETURN_NONE;
  Linear lin[3];
  for (int i = 0; i < 3; ++i)
    if (!lin[i].read(args[1 + 2 * i], args[2 + 2 * i], heads[i] * 128, K, dev)) Py_RETURN_NONE;
  OnDevice on(dev);
  at::Tensor y[3];
  int rc;
  const int64_t features = (heads[0] + 2 * heads[1]) * 128;
  bool gemm = L > 1 && L <= 0x7fffffff && K <= 65536 && xattn_proj_gemm_fits((int)L, (int)K, (int)features, 1);
  for (int i = 0; i < 3; ++i) gemm = gemm && lin[i].w->stride(0) <= (1 << 22);
  if (L == 1 || gemm) {
    const auto opts = at::TensorOptions().device(dev).dtype(at::kBFloat16);
    for (int i = 0; i < 3; ++i) y[i] = at::empty_strided({1, heads[i], L, 128}, {L * heads[i] * 128, 128, heads[i] * 128, 1}, opts);
  }
  if (L == 1) {
    rc = xattn_qkv_rope_gemv(x->data_ptr(), (int)K, lin[0].w->data_ptr(), lin[0].w->stride(0), lin[0].bias_ptr(),
                             lin[1].w->data_ptr(), lin[1].w->stride(0), lin[1].bias_ptr(), lin[2].w->data_ptr(),
                             lin[2].w->stride(0), lin[2].bias_ptr(), cos->data_ptr(), sin->data_ptr(), y[0].data_ptr(),
                             y[1].data_ptr(), y[2].data_ptr(), (int)heads[0], (int)heads[1], 128, stream_of(dev));
  } else if (gemm) {
    rc = xattn_qkv_rope_gemm(x->data_ptr(), (int)L, (int)K, lin[0].w->data_ptr(), lin[0].w->stride(0), lin[0].bias_ptr(),
                             lin[1].w->data_ptr(), lin[1].w->stride(0), lin[1].bias_ptr(), lin[2].w->data_ptr(),
                             lin[2].w->stride(0), lin[2].bias_ptr(), cos->data_ptr(), sin->data_ptr(), cos->stride(1),
                             sin->stride(1), y[0].data_ptr(), y[1].data_ptr(), y[2].data_ptr(), (int)heads[0], (int)heads[1], 128,
                             stream_of(dev));
  } else {
    for (int i = 0; i < 3; ++i) y[i] = at::linear(*x, *lin[i].w, lin[i].b);
    rc = xattn_rope(y[0].data_ptr(), y[1].data_ptr(), cos->data_ptr(), sin->data_ptr(), cos->stride(1), sin->stride(1), (int)L,
                    (int)heads[0], (int)heads[1], 128, stream_of(dev));
    for (int i = 0; i < 3; ++i)
      y[i] = y[i].as_strided({1, heads[i], L, 128}, {L * heads[i] * 128, 128, heads[i] * 128, 1});
  }
  if (rc != XATTN_OK) return fail(L == 1 ? "xattn_qkv_rope_gemv" : gemm ? "xattn_qkv_rope_gemm" : "xattn_rope", rc);
  PyObject* result = PyTuple_New(3);
  if (!result) return nullptr;
  for (int i = 0; i < 3; ++i) PyTuple_SET_ITEM(result, i, THPVariable_Wrap(std::move(y[i])));
  return result;
  END_HANDLE_TH_ERRORS
}

// output(hidden, w, b): the output projection of one token, or of as many as proj_gemm.hip takes
PyObject* output(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 3) return PyErr_Format(PyExc_TypeError, "output takes 3 arguments");
  HANDLE_TH_ERRORS
  const at::Tensor *x = hidden_of(args[0]), *w = tensor_of(args[1]);
  if (!x || !w || w->dim() != 2) Py_RETURN_NONE;
  const c10::Device dev = x->device();
  const int64_t N = w->size(0), L = x->size(1), K = x->size(2);
  Linear lin;
  if (N < 4 || N % 4 || N > 0x7fffffff || L > 0x7fffffff || !lin.read(args[1], args[2], N, K, dev)) Py_RETURN_NONE;
  if (L > 1 && (K > 65536 || lin.w->stride(0) > (1 << 22) || !xattn_proj_gemm_fits((int)L, (int)K, (int)N, 0))) Py_RETURN_NONE;
  OnDevice on(dev);
  at::Tensor y = at::empty({1, L, N}, at::TensorOptions().device(dev).dtype(at::kBFloat16));
  const int rc = L == 1 ? xattn_gemv(x->data_ptr(), (int)K, lin.w->data_ptr(), lin.w->stride(0), lin.bias_ptr(), y.data_ptr(), (int)N,
                                     stream_of(dev))
                        : xattn_gemm(x->data_ptr(), (int)L, (int)K, lin.w->data_ptr(), lin.w->stride(0), lin.bias_ptr(), y.data_ptr(),
                                     (int)N, stream_of(dev));
  if (rc != XATTN_OK) return fail(L == 1 ? "xattn_gemv" : "xattn_gemm", rc);
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyMethodDef method(const char* name) {
  return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(F)), METH_FASTCALL, nullptr};
}
PyMethodDef methods[] = {
    method<prefill>("prefill"),
    method<estimate>("estimate"),
    method<decode>("decode"),
    method<decode_layer>("decode_layer"),
    method<project>("project"),
    method<output>("output"),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "xattn_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_xattn_host(void) { return PyModule_Create(&module_def); }
