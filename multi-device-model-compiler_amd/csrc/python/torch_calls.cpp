// The package's tensor functions for the ordinary call, as a CPython extension over libtorch.
//
// A call of the package is a few checks, the output's allocation, the caller's stream and one entry
// point of the kernel library.  Done in Python through ctypes that is 5 us of interpreter and torch
// binding overhead in front of a 2.2 us kernel launch (current_stream() alone 2.5 us), more than
// most kernels of this library run; here it is 1 us (add 7.6 -> 3.9 us a call, the launch included).
//
// Every function takes positional arguments and handles the case it is written for - operands of
// the expected types and shapes, contiguous, on the current device.  Anything else returns None,
// nothing done, and the package's Python code takes over: it has the checks, the error messages and
// the rarer options (another stream).  A failure the library reports is raised here as MgpuError.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/Functions.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <initializer_list>

#include "mgpu_ops.h"

namespace {

PyObject *errorClass = nullptr; // MgpuError of the package

using at::ScalarType;
using at::Tensor;

bool is16(ScalarType t) { return t == at::kHalf || t == at::kBFloat16; }

// One call's operands: `ok` turns false at the first one outside the ordinary case.
struct Call {
  bool ok = true;
  int device;
  explicit Call(bool usable) : ok(usable), device(ok ? (int)c10::hip::current_device() : 0) {}

  const Tensor &in(PyObject *o) {
    static const Tensor none;
    if (!ok || !THPVariable_Check(o)) {
      ok = false;
      return none;
    }
    const Tensor &t = THPVariable_Unpack(o);
    ok = t.is_cuda() && t.get_device() == device && t.is_contiguous() && !t.is_conj() && !t.is_neg();
    return t;
  }
  const Tensor &in(PyObject *o, ScalarType type) {
    const Tensor &t = in(o);
    ok = ok && t.scalar_type() == type;
    return t;
  }
  // data of an operand whose shape nobody looks at (the entry points take sizes from the others)
  void *ptr(PyObject *o) {
    const Tensor &t = in(o);
    return ok ? t.data_ptr() : nullptr;
  }
  void *optional(PyObject *o) { return o == Py_None ? nullptr : ptr(o); }

  int64_t integer(PyObject *o) {
    const int64_t v = PyLong_Check(o) ? PyLong_AsLongLong(o) : (ok = false, 0);
    if (v == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      ok = false;
    }
    return v;
  }
  int32_t integer32(PyObject *o) {
    const int64_t v = integer(o);
    if (v != (int32_t)v) ok = false;
    return (int32_t)v;
  }
  float real(PyObject *o) {
    if (PyFloat_CheckExact(o)) return (float)PyFloat_AS_DOUBLE(o);
    ok = false;
    return 0.0f;
  }
  // the softmax scale; None: 1 / sqrt(head size), rounded as Python's float is on its way into a C float
  float scale(PyObject *o, int32_t headDim) {
    return o == Py_None ? (float)(1.0 / std::sqrt((double)headDim)) : real(o);
  }
  bool flag(PyObject *o) {
    if (!PyBool_Check(o)) ok = false;
    return o == Py_True;
  }
  int32_t size32(int64_t v) {
    if (v != (int32_t)v) ok = false;
    return (int32_t)v;
  }

  Tensor empty(at::IntArrayRef shape, ScalarType type) const {
    return Tensor(at::detail::empty_cuda(shape, type, at::Device(at::kCUDA, (c10::DeviceIndex)device), std::nullopt));
  }
  mgpuStream_t stream() const { return c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }
};

// Runs one entry point (the interpreter free meanwhile, as under ctypes) and hands out its outputs.
template <typename F> bool launched(F &&f) {
  const char *message;
  Py_BEGIN_ALLOW_THREADS
  f();
  message = mgpuOpsTakeLastError();
  Py_END_ALLOW_THREADS
  if (!message) return true;
  PyErr_SetString(errorClass ? errorClass : PyExc_RuntimeError, message);
  return false;
}

PyObject *wrap(Tensor t) { return THPVariable_Wrap(std::move(t)); }

PyObject *wrap(std::initializer_list<Tensor> ts) {
  PyObject *tuple = PyTuple_New((Py_ssize_t)ts.size());
  if (!tuple) return nullptr;
  Py_ssize_t i = 0;
  for (const Tensor &t : ts) {
    PyObject *o = THPVariable_Wrap(t);
    if (!o) {
      Py_DECREF(tuple);
      return nullptr;
    }
    PyTuple_SET_ITEM(tuple, i++, o);
  }
  return tuple;
}

PyObject *same(PyObject *o) {
  Py_INCREF(o);
  return o;
}

#define MDMC_CALL(NAME, COUNT)                                              \
  PyObject *NAME##Impl(PyObject *const *a, Call &c);                        \
  PyObject *NAME(PyObject *, PyObject *const *a, Py_ssize_t n) {            \
    HANDLE_TH_ERRORS                                                        \
    Call c(n == COUNT);                                                     \
    if (!c.ok) Py_RETURN_NONE;                                              \
    return NAME##Impl(a, c);                                                \
    END_HANDLE_TH_ERRORS                                                    \
  }                                                                         \
  PyObject *NAME##Impl(PyObject *const *a, Call &c)

// add(a, b, out | None)
MDMC_CALL(add, 3) {
  const Tensor &x = c.in(a[0], at::kFloat), &y = c.in(a[1], at::kFloat);
  if (!c.ok || x.sizes() != y.sizes()) Py_RETURN_NONE;
  Tensor fresh;
  float *dst;
  if (a[2] == Py_None) {
    fresh = c.empty(x.sizes(), at::kFloat);
    dst = static_cast<float *>(fresh.data_ptr());
  } else {
    dst = static_cast<float *>(c.ptr(a[2]));
    if (!c.ok) Py_RETURN_NONE;
  }
  const mgpuStream_t s = c.stream();
  const auto *px = static_cast<const float *>(x.data_ptr()), *py = static_cast<const float *>(y.data_ptr());
  const int64_t n = x.numel();
  if (!launched([&] { mgpuAddF32(px, py, dst, n, s); })) return nullptr;
  return a[2] == Py_None ? wrap(std::move(fresh)) : same(a[2]);
}

struct Rows {
  int32_t m = 0, n = 0;
};
Rows rowsOf(Call &c, const Tensor &x) {
  Rows r;
  if (!c.ok || x.dim() == 0) {
    c.ok = false;
    return r;
  }
  r.n = c.size32(x.size(-1));
  r.m = c.size32(r.n ? x.numel() / r.n : 0);
  return r;
}

// layer_norm(x, gamma, beta, eps, out | None)
MDMC_CALL(layer_norm, 5) {
  const Tensor &x = c.in(a[0]);
  const Rows r = rowsOf(c, x);
  if (!c.ok) Py_RETURN_NONE;
  const ScalarType t = x.scalar_type();
  if (t != at::kFloat && !is16(t)) Py_RETURN_NONE;
  const void *gamma = c.ptr(a[1]), *beta = c.ptr(a[2]);
  const float eps = c.real(a[3]);
  void *dst = c.optional(a[4]);
  if (!c.ok) Py_RETURN_NONE;
  Tensor fresh;
  if (!dst && a[4] == Py_None) {
    fresh = c.empty(x.sizes(), t);
    dst = fresh.data_ptr();
  }
  const mgpuStream_t s = c.stream();
  const void *in = x.data_ptr();
  const bool fine = launched([&] {
    if (t == at::kFloat)
      mgpuLayerNormF32((const float *)in, (const float *)gamma, (const float *)beta, (float *)dst, eps, r.m, r.n, s);
    else if (t == at::kHalf) mgpuLayerNormF16(in, gamma, beta, dst, eps, r.m, r.n, s);
    else mgpuLayerNormBF16(in, gamma, beta, dst, eps, r.m, r.n, s);
  });
  if (!fine) return nullptr;
  return a[4] == Py_None ? wrap(std::move(fresh)) : same(a[4]);
}

// cast_layer_norm(x, gamma, beta, eps) -> (cast, normed)
MDMC_CALL(cast_layer_norm, 4) {
  const Tensor &x = c.in(a[0], at::kFloat);
  const Rows r = rowsOf(c, x);
  const void *gamma = c.ptr(a[1]), *beta = c.ptr(a[2]);
  const float eps = c.real(a[3]);
  if (!c.ok) Py_RETURN_NONE;
  Tensor cast = c.empty(x.sizes(), at::kHalf), normed = c.empty(x.sizes(), at::kHalf);
  const mgpuStream_t s = c.stream();
  const auto *in = static_cast<const float *>(x.data_ptr());
  void *pc = cast.data_ptr(), *pn = normed.data_ptr();
  if (!launched([&] { mgpuCastLayerNormF32ToF16(in, gamma, beta, pc, pn, eps, r.m, r.n, s); })) return nullptr;
  return wrap({cast, normed});
}

// add_residual_layer_norm(x, residual, gamma, beta, eps) -> (summed, normed)
MDMC_CALL(add_residual_layer_norm, 5) {
  const Tensor &x = c.in(a[0]);
  const Rows r = rowsOf(c, x);
  if (!c.ok) Py_RETURN_NONE;
  const ScalarType t = x.scalar_type();
  if (t != at::kFloat && !is16(t)) Py_RETURN_NONE;
  const void *residual = c.ptr(a[1]), *gamma = c.ptr(a[2]), *beta = c.ptr(a[3]);
  const float eps = c.real(a[4]);
  if (!c.ok) Py_RETURN_NONE;
  Tensor summed = c.empty(x.sizes(), t), normed = c.empty(x.sizes(), t);
  const mgpuStream_t s = c.stream();
  const void *in = x.data_ptr();
  void *ps = summed.data_ptr(), *pn = normed.data_ptr();
  const bool fine = launched([&] {
    if (t == at::kFloat)
      mgpuAddResidualPreLayerNormF32((const float *)in, (const float *)residual, (const float *)gamma, (const float *)beta,
                                     (float *)ps, (float *)pn, eps, r.m, r.n, s);
    else if (t == at::kHalf) mgpuAddResidualPreLayerNormF16(in, residual, gamma, beta, ps, pn, eps, r.m, r.n, s);
    else mgpuAddResidualPreLayerNormBF16(in, residual, gamma, beta, ps, pn, eps, r.m, r.n, s);
  });
  if (!fine) return nullptr;
  return wrap({summed, normed});
}

// fused_mha(qkv, seqlens | None, scale | None, causal, out | None)
MDMC_CALL(fused_mha, 5) {
  const Tensor &qkv = c.in(a[0]);
  if (!c.ok || !is16(qkv.scalar_type()) || qkv.dim() != 5 || qkv.size(2) != 3) Py_RETURN_NONE;
  const int32_t B = c.size32(qkv.size(0)), S = c.size32(qkv.size(1)), H = c.size32(qkv.size(3)), D = c.size32(qkv.size(4));
  const int32_t *lens = nullptr;
  if (a[1] != Py_None) {
    const Tensor &l = c.in(a[1], at::kInt);
    if (!c.ok || l.numel() != B) Py_RETURN_NONE;
    lens = static_cast<const int32_t *>(l.data_ptr());
  }
  const float scale = c.scale(a[2], D);
  const bool causal = c.flag(a[3]);
  void *dst = c.optional(a[4]);
  if (!c.ok) Py_RETURN_NONE;
  Tensor fresh;
  if (!dst && a[4] == Py_None) {
    fresh = c.empty({B, S, (int64_t)H * D}, qkv.scalar_type());
    dst = fresh.data_ptr();
  }
  const mgpuStream_t s = c.stream();
  const void *in = qkv.data_ptr();
  const bool half = qkv.scalar_type() == at::kHalf;
  if (!launched([&] { (half ? mgpuFusedMHAF16 : mgpuFusedMHABF16)(in, lens, dst, B, S, H, D, scale, causal, s); })) return nullptr;
  return a[4] == Py_None ? wrap(std::move(fresh)) : same(a[4]);
}

// fused_mha_cu_seqlens(qkv, cu_seqlens, max_s, scale | None, causal, out | None)
MDMC_CALL(fused_mha_cu_seqlens, 6) {
  const Tensor &qkv = c.in(a[0]), &cu = c.in(a[1], at::kInt);
  if (!c.ok || !is16(qkv.scalar_type()) || qkv.dim() != 4 || qkv.size(1) != 3) Py_RETURN_NONE;
  const int32_t B = c.size32(cu.numel() - 1), maxS = c.integer32(a[2]), H = c.size32(qkv.size(2)), D = c.size32(qkv.size(3));
  const float scale = c.scale(a[3], D);
  const bool causal = c.flag(a[4]);
  void *dst = c.optional(a[5]);
  if (!c.ok) Py_RETURN_NONE;
  Tensor fresh;
  if (!dst && a[5] == Py_None) {
    fresh = c.empty({qkv.size(0), (int64_t)H * D}, qkv.scalar_type());
    dst = fresh.data_ptr();
  }
  const mgpuStream_t s = c.stream();
  const void *in = qkv.data_ptr();
  const auto *lens = static_cast<const int32_t *>(cu.data_ptr());
  const bool half = qkv.scalar_type() == at::kHalf;
  if (!launched([&] { (half ? mgpuFusedMHAF16CuSeqlens : mgpuFusedMHABF16CuSeqlens)(in, lens, dst, B, maxS, H, D, scale, causal, s); }))
    return nullptr;
  return a[5] == Py_None ? wrap(std::move(fresh)) : same(a[5]);
}

template <ScalarType FROM, ScalarType TO, typename F> PyObject *castCall(PyObject *const *a, Call &c, F entry) {
  const Tensor &x = c.in(a[0], FROM);
  if (!c.ok) Py_RETURN_NONE;
  Tensor out = c.empty(x.sizes(), TO);
  const mgpuStream_t s = c.stream();
  void *src = x.data_ptr(), *dst = out.data_ptr();
  const size_t n = (size_t)x.numel();
  if (!launched([&] { entry(dst, src, n, s); })) return nullptr;
  return wrap(std::move(out));
}
MDMC_CALL(cast_f32_to_f16, 1) {
  return castCall<at::kFloat, at::kHalf>(a, c, [](void *d, void *s, size_t n, mgpuStream_t q) { mgpuCastF32ToF16(d, (const float *)s, n, q); });
}
MDMC_CALL(cast_f16_to_f32, 1) {
  return castCall<at::kHalf, at::kFloat>(a, c, [](void *d, void *s, size_t n, mgpuStream_t q) { mgpuCastF16ToF32((float *)d, s, n, q); });
}
MDMC_CALL(cast_f32_to_bf16, 1) {
  return castCall<at::kFloat, at::kBFloat16>(a, c, [](void *d, void *s, size_t n, mgpuStream_t q) { mgpuCastF32ToBF16(d, (const float *)s, n, q); });
}
MDMC_CALL(cast_bf16_to_f32, 1) {
  return castCall<at::kBFloat16, at::kFloat>(a, c, [](void *d, void *s, size_t n, mgpuStream_t q) { mgpuCastBF16ToF32((float *)d, s, n, q); });
}

// qkv_bias_transpose(qkv, bias | None) -> (q, k, v)
MDMC_CALL(qkv_bias_transpose, 2) {
  const Tensor &qkv = c.in(a[0]);
  void *bias = c.optional(a[1]);
  if (!c.ok || !is16(qkv.scalar_type()) || qkv.dim() != 5) Py_RETURN_NONE;
  const int32_t B = c.size32(qkv.size(0)), S = c.size32(qkv.size(1)), H = c.size32(qkv.size(3)), D = c.size32(qkv.size(4));
  const int32_t tokens = c.size32((int64_t)B * S);
  if (!c.ok) Py_RETURN_NONE;
  const ScalarType t = qkv.scalar_type();
  Tensor q = c.empty({B, H, S, D}, t), k = c.empty({B, H, S, D}, t), v = c.empty({B, H, S, D}, t);
  const mgpuStream_t s = c.stream();
  void *in = qkv.data_ptr(), *pq = q.data_ptr(), *pk = k.data_ptr(), *pv = v.data_ptr();
  const bool fine = launched([&] {
    (t == at::kHalf ? mgpuAddFusedQKVBiasTransposeF16 : mgpuAddFusedQKVBiasTransposeBF16)(pq, pk, pv, in, bias, B, S, tokens, H, D, s);
  });
  if (!fine) return nullptr;
  return wrap({q, k, v});
}

// matmul_ex(x, w, bias | None, residual | None, act, packed)
MDMC_CALL(matmul_ex, 6) {
  const Tensor &x = c.in(a[0]), &w = c.in(a[1]);
  if (!c.ok || x.dim() != 2 || w.dim() != 2) Py_RETURN_NONE;
  const ScalarType t = x.scalar_type();
  void *bias = c.optional(a[2]), *residual = c.optional(a[3]);
  const int32_t act = c.integer32(a[4]);
  const bool packed = c.flag(a[5]);
  if (!c.ok || (t != at::kFloat && !is16(t)) || (packed && t == at::kFloat)) Py_RETURN_NONE;
  const int64_t M = x.size(0), K = x.size(1), N = w.size(packed ? 0 : 1);
  if (w.size(packed ? 1 : 0) != K) Py_RETURN_NONE;
  Tensor out = c.empty({M, N}, t);
  const mgpuStream_t s = c.stream();
  void *in = x.data_ptr(), *pw = w.data_ptr(), *dst = out.data_ptr();
  const bool fine = launched([&] {
    if (t == at::kFloat)
      mgpuMatmulExF32((float *)in, (float *)pw, (float *)bias, (float *)dst, (float *)residual, M, N, K, bias != nullptr, act,
                      residual != nullptr, s);
    else
      (t == at::kHalf ? (packed ? mgpuMatmulExPackedF16 : mgpuMatmulExF16) : (packed ? mgpuMatmulExPackedBF16 : mgpuMatmulExBF16))(
          in, pw, bias, dst, residual, M, N, K, bias != nullptr, act, residual != nullptr, s);
  });
  if (!fine) return nullptr;
  return wrap(std::move(out));
}

int64_t convOut(int64_t size, int64_t k, int64_t lead, int64_t trail, int64_t stride, int64_t dilation) {
  const int64_t span = size + lead + trail - dilation * (k - 1) - 1;
  return span < 0 || stride < 1 ? -1 : span / stride + 1;
}

bool integers(Call &c, PyObject *o, int64_t *v, Py_ssize_t count) {
  if (!PyTuple_Check(o) || PyTuple_GET_SIZE(o) != count) c.ok = false;
  for (Py_ssize_t i = 0; c.ok && i < count; i++) v[i] = c.integer(PyTuple_GET_ITEM(o, i));
  return c.ok;
}

// conv2d(x, w, bias, post_add | None, pad, stride, dilation, relu)
MDMC_CALL(conv2d, 8) {
  const Tensor &x = c.in(a[0], at::kFloat), &w = c.in(a[1], at::kFloat);
  void *bias = c.ptr(a[2]), *post = c.optional(a[3]);
  int64_t pad[4], st[2], di[2];
  if (!integers(c, a[4], pad, 4) || !integers(c, a[5], st, 2) || !integers(c, a[6], di, 2)) Py_RETURN_NONE;
  const bool relu = c.flag(a[7]);
  if (!c.ok || x.dim() != 4 || w.dim() != 4 || x.size(1) != w.size(1)) Py_RETURN_NONE;
  const int64_t N = x.size(0), IC = x.size(1), H = x.size(2), W = x.size(3), OC = w.size(0), KH = w.size(2), KW = w.size(3);
  const int64_t OH = convOut(H, KH, pad[0], pad[2], st[0], di[0]), OW = convOut(W, KW, pad[1], pad[3], st[1], di[1]);
  if (OH < 0 || OW < 0) Py_RETURN_NONE;
  Tensor out = c.empty({N, OC, OH, OW}, at::kFloat);
  const mgpuStream_t s = c.stream();
  auto *in = static_cast<float *>(x.data_ptr()), *pw = static_cast<float *>(w.data_ptr()), *dst = static_cast<float *>(out.data_ptr());
  const bool fine = launched([&] {
    mgpuConv2d(in, pw, (float *)bias, dst, (float *)post, N, IC, H, W, OC, KH, KW, OH, OW, pad[0], pad[1], pad[2], pad[3], st[0], st[1],
               di[0], di[1], post != nullptr, relu, s);
  });
  if (!fine) return nullptr;
  return wrap(std::move(out));
}

// pool2d(x, kernel, pad, stride, average)
MDMC_CALL(pool2d, 5) {
  const Tensor &x = c.in(a[0], at::kFloat);
  int64_t k[2], pad[4], st[2];
  if (!integers(c, a[1], k, 2) || !integers(c, a[2], pad, 4) || !integers(c, a[3], st, 2)) Py_RETURN_NONE;
  const bool average = c.flag(a[4]);
  if (!c.ok || x.dim() != 4) Py_RETURN_NONE;
  const int64_t N = x.size(0), C = x.size(1), H = x.size(2), W = x.size(3);
  const int64_t OH = convOut(H, k[0], pad[0], pad[2], st[0], 1), OW = convOut(W, k[1], pad[1], pad[3], st[1], 1);
  if (OH < 0 || OW < 0) Py_RETURN_NONE;
  Tensor out = c.empty({N, C, OH, OW}, at::kFloat);
  const mgpuStream_t s = c.stream();
  auto *in = static_cast<float *>(x.data_ptr()), *dst = static_cast<float *>(out.data_ptr());
  const bool fine = launched([&] {
    mgpuPool2d(in, dst, N, C, H, W, OH, OW, k[0], k[1], pad[0], pad[1], pad[2], pad[3], st[0], st[1], average ? 1 : 0, s);
  });
  if (!fine) return nullptr;
  return wrap(std::move(out));
}

// decoding_context_layer(x, wqkv, wo, bo, w1, b1, w2, b2, heads, causal, relu, norm_first)
MDMC_CALL(decoding_context_layer, 12) {
  const Tensor &x = c.in(a[0], at::kFloat);
  if (!c.ok || x.dim() != 3) Py_RETURN_NONE;
  float *w[7];
  for (int i = 0; i < 7; i++) w[i] = static_cast<float *>(c.ptr(a[1 + i]));
  const int64_t heads = c.integer(a[8]);
  const bool causal = c.flag(a[9]), relu = c.flag(a[10]), normFirst = c.flag(a[11]);
  if (!c.ok) Py_RETURN_NONE;
  const Tensor &w1 = THPVariable_Unpack(a[4]);
  if (w1.dim() < 2) Py_RETURN_NONE;
  const int64_t B = x.size(0), S = x.size(1), d = x.size(2), ffn = w1.size(1);
  Tensor out = c.empty(x.sizes(), at::kFloat);
  const mgpuStream_t s = c.stream();
  auto *in = static_cast<float *>(x.data_ptr()), *dst = static_cast<float *>(out.data_ptr());
  const bool fine = launched([&] {
    mgpuLLMDecodingContextLayer(in, w[0], w[1], w[2], w[3], w[4], w[5], w[6], dst, B, S, d, ffn, heads, normFirst, causal, relu, s);
  });
  if (!fine) return nullptr;
  return wrap(std::move(out));
}

// bert_encoder_layer(x, wqkv, bqkv, wo, bo, g1, be1, w1, b1, w2, b2, g2, be2, heads, seqlens | None, eps, out | None, no_alloc)
MDMC_CALL(bert_encoder_layer, 18) {
  const Tensor &x = c.in(a[0]);
  if (!c.ok || x.dim() != 3) Py_RETURN_NONE;
  const void *w[12];
  for (int i = 0; i < 12; i++) w[i] = c.ptr(a[1 + i]);
  const int64_t heads = c.integer(a[13]);
  const auto *lens = static_cast<const int32_t *>(c.optional(a[14]));
  const float eps = c.real(a[15]);
  void *dst = c.optional(a[16]);
  const bool noAlloc = c.flag(a[17]);
  if (!c.ok) Py_RETURN_NONE;
  const Tensor &w1 = THPVariable_Unpack(a[7]);
  if (w1.dim() < 2) Py_RETURN_NONE;
  const int64_t B = x.size(0), S = x.size(1), d = x.size(2), ffn = w1.size(1);
  Tensor fresh;
  if (!dst && a[16] == Py_None) {
    fresh = c.empty(x.sizes(), x.scalar_type());
    dst = fresh.data_ptr();
  }
  const mgpuStream_t s = c.stream();
  const void *in = x.data_ptr();
  const bool fine = launched([&] {
    (noAlloc ? mgpuBertEncoderLayerF16NoAlloc : mgpuBertEncoderLayerF16)(in, w[0], w[1], w[2], w[3], w[4], w[5], w[6], w[7], w[8], w[9], w[10],
                                                                         w[11], lens, dst, B, S, d, ffn, heads, eps, s);
  });
  if (!fine) return nullptr;
  return a[16] == Py_None ? wrap(std::move(fresh)) : same(a[16]);
}

// set_error(cls): what a failure of the library is raised as
PyObject *set_error(PyObject *, PyObject *const *a, Py_ssize_t n) {
  if (n != 1) {
    PyErr_SetString(PyExc_TypeError, "set_error takes the exception class");
    return nullptr;
  }
  Py_INCREF(a[0]);
  Py_XDECREF(errorClass);
  errorClass = a[0];
  Py_RETURN_NONE;
}

#define MDMC_METHOD(NAME) {#NAME, (PyCFunction)(void (*)(void))NAME, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {MDMC_METHOD(set_error),
                         MDMC_METHOD(add),
                         MDMC_METHOD(layer_norm),
                         MDMC_METHOD(cast_layer_norm),
                         MDMC_METHOD(add_residual_layer_norm),
                         MDMC_METHOD(fused_mha),
                         MDMC_METHOD(fused_mha_cu_seqlens),
                         MDMC_METHOD(cast_f32_to_f16),
                         MDMC_METHOD(cast_f16_to_f32),
                         MDMC_METHOD(cast_f32_to_bf16),
                         MDMC_METHOD(cast_bf16_to_f32),
                         MDMC_METHOD(qkv_bias_transpose),
                         MDMC_METHOD(matmul_ex),
                         MDMC_METHOD(conv2d),
                         MDMC_METHOD(pool2d),
                         MDMC_METHOD(decoding_context_layer),
                         MDMC_METHOD(bert_encoder_layer),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "mdmc_torch_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit_mdmc_torch_calls(void) { return PyModule_Create(&module); }
