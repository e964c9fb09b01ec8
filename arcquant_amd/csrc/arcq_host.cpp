// arcq_host.cpp -- the Python operators' way to the C ABI of libarcq_hip.so for the ordinary case: argument checks, output
// tensors from torch's allocator, torch's current stream and the launch, in one native call.
//
// A decode step is a chain of launches of a few microseconds each, and through Python and ctypes an operator costs the host 8
// to 14 us (fused norm + quantizer of one row 12.4 us a call, 6.9 so; decode step of a layer, MXFP4, 8 sequences 169 us, 85 so).
//
// Every function here returns None, with no error set and nothing launched, for arguments it does not take: wrong types,
// shapes, devices or alignments, tensor subclasses and wrapped tensors, active dispatch or function modes, no memory, and any status the
// library refuses them with.  The Python operator then runs its own checks and raises what it always raised, or computes the
// call by the general route.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <limits.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>

#include "../../include/arcq.h"

namespace {

struct NotTaken {};  // thrown by the checks below, caught at the entry

void need(bool ok) {
  if (!ok) throw NotTaken();
}

// a plain GPU tensor: no subclass, no functorch or Python wrapper around it
const at::Tensor &tensor(PyObject *o) {
  need(THPVariable_CheckExact(o));
  const at::Tensor &t = THPVariable_Unpack(o);
  need(t.defined() && t.is_cuda() && t.layout() == at::kStrided);
  const c10::DispatchKeySet ks = t.key_set();
  need(!ks.has(c10::DispatchKey::Python) && !ks.has(c10::DispatchKey::FuncTorchBatched) &&
       !ks.has(c10::DispatchKey::FuncTorchGradWrapper) && !ks.has(c10::DispatchKey::Functionalize) && !t.is_neg() && !t.is_conj());
  return t;
}

const at::Tensor &tensor(PyObject *o, at::ScalarType type, int64_t dims = -1) {
  const at::Tensor &t = tensor(o);
  need(t.scalar_type() == type && (dims < 0 || t.dim() == dims) && t.is_contiguous());
  return t;
}

// bf16 [M, K], unit stride along K, rows possibly strided
const at::Tensor &rows(PyObject *o) {
  const at::Tensor &t = tensor(o);
  need(t.scalar_type() == at::kBFloat16 && t.dim() == 2 && t.stride(1) == 1);
  return t;
}

int as_int(int64_t v) {
  need(v >= 0 && v <= INT_MAX);
  return (int)v;
}

int number(PyObject *o) {
  need(PyLong_CheckExact(o));
  const long v = PyLong_AsLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    throw NotTaken();
  }
  return as_int(v);
}

double real(PyObject *o) {
  need(PyFloat_CheckExact(o) || PyLong_CheckExact(o));
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    throw NotTaken();
  }
  return v;
}

int format(PyObject *o) {
  need(PyUnicode_CheckExact(o));
  if (PyUnicode_CompareWithASCIIString(o, "NVFP4") == 0) return ARCQ_FMT_NVFP4;
  need(PyUnicode_CompareWithASCIIString(o, "MXFP4") == 0);
  return ARCQ_FMT_MXFP4;
}

bool is_absmax(PyObject *o) {
  if (!PyUnicode_CheckExact(o)) return false;
  need(PyUnicode_CompareWithASCIIString(o, "absmax") == 0);
  return true;
}

// None, a number, or one fp32 value on the operands' device
struct Scale {
  double host = 1.0;
  const float *device = nullptr;
};
Scale scale(PyObject *o, const at::Device &dev) {
  Scale s;
  if (o == Py_None) return s;
  if (PyFloat_CheckExact(o) || PyLong_CheckExact(o)) {
    s.host = real(o);
    return s;
  }
  const at::Tensor &t = tensor(o);
  need(t.scalar_type() == at::kFloat && t.numel() == 1 && t.device() == dev);
  s.device = t.const_data_ptr<float>();
  return s;
}

at::Tensor empty(at::IntArrayRef shape, const at::Tensor &like, at::ScalarType type) {
  return at::empty(shape, at::TensorOptions().dtype(type).device(like.device()));
}

void *stream(const at::Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// the launch, with t's device current and other Python threads free to run
template <class F>
void launch(const at::Tensor &t, F f) {
  const c10::DeviceGuard guard(t.device());
  void *st = stream(t);
  int rc;
  Py_BEGIN_ALLOW_THREADS rc = f(st);
  Py_END_ALLOW_THREADS need(rc == ARCQ_OK);
}

PyObject *pack(std::initializer_list<at::Tensor> ts) {
  PyObject *r = PyTuple_New((Py_ssize_t)ts.size());
  if (!r) return nullptr;
  Py_ssize_t i = 0;
  for (const at::Tensor &t : ts) {
    PyObject *o = THPVariable_Wrap(t);
    if (!o) {
      Py_DECREF(r);
      return nullptr;
    }
    PyTuple_SET_ITEM(r, i++, o);
  }
  return r;
}

// the quantizers' conditions on K, select_num and the outputs
struct Quantized {
  at::Tensor codes, scales;
  Quantized(const at::Tensor &x, int M, int K, const at::Tensor &index, int KE, int fmt) {
    const int G = fmt == ARCQ_FMT_NVFP4 ? 16 : 32;
    need(index.numel() == K && index.device() == x.device());
    need(K % 32 == 0 && K >= 32 && K <= 32736 && KE <= K && KE % G == 0);
    codes = empty({M, (K + KE) / 2}, x, at::kByte);
    scales = empty({(int64_t)M * ((K + KE) / G)}, x, at::kByte);
  }
};

// (kind, X, gamma, eps, reorder_index, KE, fmt, global_scale); kind 0: activations, 1: weights, 2: fused RMSNorm
PyObject *quantize(PyObject *const *a) {
  const int kind = number(a[0]);
  const at::Tensor &x = tensor(a[1], at::kBFloat16, 2), &index = tensor(a[4], at::kShort, 1);
  const int M = as_int(x.size(0)), K = as_int(x.size(1)), KE = number(a[5]), fmt = format(a[6]);
  const bool absmax = is_absmax(a[7]);
  need(!absmax || kind == 0);
  const Scale gs = absmax ? Scale() : scale(a[7], x.device());
  const at::Tensor *gamma = nullptr;
  float eps = 0.0f;
  if (kind == 2) {
    gamma = &tensor(a[2], at::kBFloat16, 1);
    need(gamma->numel() == K && gamma->device() == x.device());
    eps = (float)real(a[3]);
  }
  const Quantized q(x, M, K, index, KE, fmt);
  const at::Tensor out = absmax ? empty({}, x, at::kFloat) : at::Tensor();
  const void *xp = x.const_data_ptr();
  const int16_t *ip = index.const_data_ptr<int16_t>();
  void *cp = q.codes.data_ptr(), *sp = q.scales.data_ptr();
  launch(x, [&](void *st) {
    if (absmax)
      return arcq_reorder_quantize_x_absmax(xp, M, K, ip, KE, fmt, 2688.0f, static_cast<float *>(out.data_ptr()), cp, sp, st);
    if (kind == 2)
      return arcq_rmsnorm_quantize_x(xp, gamma->const_data_ptr(), eps, M, K, ip, KE, fmt, (float)gs.host, gs.device, cp, sp,
                                     st);
    const auto f = kind == 0 ? arcq_reorder_quantize_x : arcq_reorder_quantize_w;
    return f(xp, M, K, ip, KE, fmt, (float)gs.host, gs.device, cp, sp, st);
  });
  return absmax ? pack({q.codes, q.scales, out}) : pack({q.codes, q.scales});
}

// (gate, up, reorder_index, KE, fmt, global_scale)
PyObject *swiglu_quantize(PyObject *const *a) {
  const at::Tensor &gate = rows(a[0]), &up = rows(a[1]), &index = tensor(a[2], at::kShort, 1);
  need(gate.sizes() == up.sizes() && gate.stride(0) == up.stride(0) && gate.device() == up.device());
  const int M = as_int(gate.size(0)), K = as_int(gate.size(1)), KE = number(a[3]), fmt = format(a[4]);
  const int ld = as_int(M > 1 ? gate.stride(0) : K);
  need(ld % 8 == 0);
  const bool absmax = is_absmax(a[5]);
  const at::Tensor out = absmax ? empty({}, gate, at::kFloat) : at::Tensor();
  Scale gs = absmax ? Scale() : scale(a[5], gate.device());
  if (absmax) gs.device = out.const_data_ptr<float>();
  const Quantized q(gate, M, K, index, KE, fmt);
  const void *gp = gate.const_data_ptr(), *up_ = up.const_data_ptr();
  const int16_t *ip = index.const_data_ptr<int16_t>();
  void *cp = q.codes.data_ptr(), *sp = q.scales.data_ptr();
  launch(gate, [&](void *st) {
    if (absmax) {
      const int rc = arcq_tensor_scale(gp, up_, ld, M, K, 2688.0f, static_cast<float *>(out.data_ptr()), st);
      if (rc != ARCQ_OK) return rc;
    }
    return arcq_swiglu_quantize_x(gp, up_, ld, M, K, ip, KE, fmt, (float)gs.host, gs.device, cp, sp, st);
  });
  return absmax ? pack({q.codes, q.scales, out}) : pack({q.codes, q.scales});
}

// (A, B, SFA, SFB, scale, fmt or None, residual or None); a product that wants scratch memory of the caller's is not taken
PyObject *matmul(PyObject *const *a) {
  const at::Tensor &A = tensor(a[0], at::kByte, 2), &B = tensor(a[1], at::kByte, 2);
  const at::Tensor &SFA = tensor(a[2], at::kByte), &SFB = tensor(a[3], at::kByte);
  need(A.size(1) == B.size(1) && A.device() == B.device() && A.device() == SFA.device() && A.device() == SFB.device());
  const int M = as_int(A.size(0)), N = as_int(B.size(0)), Kp = as_int(2 * A.size(1));
  int fmt;
  if (a[5] == Py_None) {
    fmt = SFA.numel() == (int64_t)M * (Kp / 16) ? ARCQ_FMT_NVFP4 : ARCQ_FMT_MXFP4;
  } else {
    fmt = format(a[5]);
  }
  const int G = fmt == ARCQ_FMT_NVFP4 ? 16 : 32;
  need(SFA.numel() == (int64_t)M * (Kp / G) && SFB.numel() == (int64_t)N * (Kp / G) && Kp % 64 == 0);
  Scale sa, sb;
  if (PyTuple_CheckExact(a[4])) {
    need(PyTuple_GET_SIZE(a[4]) == 2);
    sa = scale(PyTuple_GET_ITEM(a[4], 0), A.device());
    sb = scale(PyTuple_GET_ITEM(a[4], 1), A.device());
  } else {
    sa = scale(a[4], A.device());
  }
  const at::Tensor *res = nullptr;
  if (a[6] != Py_None) {
    res = &tensor(a[6], at::kBFloat16, 2);
    need(res->size(0) == M && res->size(1) == N && res->device() == A.device());
  }
  need(!(M > 64 && fmt == ARCQ_FMT_NVFP4 && arcq_gemm_scratch_bytes(M, N, Kp, fmt, 0)));
  const at::Tensor C = empty({M, N}, A, at::kBFloat16);
  const void *ap = A.const_data_ptr(), *bp = B.const_data_ptr(), *asp = SFA.const_data_ptr(), *bsp = SFB.const_data_ptr();
  const float alpha = (float)(sa.host * sb.host);
  void *cp = C.data_ptr();
  launch(A, [&](void *st) {
    if (res) return arcq_matmul_add(ap, asp, bp, bsp, M, N, Kp, fmt, alpha, sa.device, sb.device, res->const_data_ptr(), cp, st);
    return arcq_matmul(ap, asp, bp, bsp, M, N, Kp, fmt, alpha, sa.device, sb.device, cp, st);
  });
  return THPVariable_Wrap(C);
}

// (qkv, query heads, cos, sin, positions, pages, params, indptr, indices, last_page_offset, layer): the rotary embedding and quantized append
// of one new token per sequence, then the attention over the pages -> [batch, query heads * 128]
PyObject *decode_step(PyObject *const *a) {
  const at::Tensor &qkv = tensor(a[0]), &cos = tensor(a[2]), &sin = tensor(a[3]);
  const at::Tensor &pos = tensor(a[4], at::kInt), &pages = tensor(a[5], at::kByte, 6), &params = tensor(a[6]);
  const at::Tensor &indptr = tensor(a[7], at::kInt), &indices = tensor(a[8], at::kInt), &last = tensor(a[9], at::kInt);
  const int nqo = number(a[1]), layer = number(a[10]);
  const at::ScalarType type = params.scalar_type();
  need((type == at::kHalf || type == at::kBFloat16) && params.dim() == 6 && params.is_contiguous());
  const int layers = as_int(pages.size(1)), heads = as_int(pages.size(3)), page = as_int(pages.size(4)), dim = as_int(2 * pages.size(5));
  const int batch = as_int(last.numel()), dt = type == at::kHalf ? 0 : 1;
  need(qkv.dim() == 2 && qkv.size(0) == batch && qkv.scalar_type() == type && qkv.stride(1) == 1 && qkv.size(1) >= ((int64_t)nqo + 2 * heads) * dim);
  for (const at::Tensor *t : {&cos, &sin})
    need(t->scalar_type() == type && t->dim() == 2 && t->size(1) == dim / 2 && t->is_contiguous());
  need(cos.size(0) == sin.size(0) && pos.numel() == batch);
  for (const at::Tensor *t : {&cos, &sin, &pos, &pages, &params, &indptr, &indices, &last}) need(t->device() == qkv.device());
  const at::Tensor q = empty({batch, nqo, dim}, qkv, type), out = empty({batch, (int64_t)nqo * dim}, qkv, type);
  const int ld = as_int(qkv.stride(0)), table = as_int(cos.size(0));
  const float sm = (float)(1.0 / std::sqrt((double)dim));
  const int32_t *ip = indptr.const_data_ptr<int32_t>(), *xp = indices.const_data_ptr<int32_t>(), *lp = last.const_data_ptr<int32_t>();
  void *pg = pages.data_ptr(), *pr = params.data_ptr(), *qp = q.data_ptr(), *op = out.data_ptr();
  launch(qkv, [&](void *st) {
    const int rc = arcq_rope_kv_append_i4(qkv.const_data_ptr(), ld, dt, batch, nqo, cos.const_data_ptr(), sin.const_data_ptr(), table,
                                          pos.const_data_ptr<int32_t>(), qp, pg, pr, ip, xp, lp, layers, layer, heads, page, dim, st);
    if (rc != ARCQ_OK) return rc;
    return arcq_kv_decode_i4(op, qp, dt, batch, nqo, pg, pr, ip, xp, lp, layers, layer, heads, page, dim, sm, st);
  });
  return THPVariable_Wrap(out);
}

template <PyObject *(*F)(PyObject *const *), int N>
PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != N) {
    PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", N, n);
    return nullptr;
  }
  try {
    if (!c10::impl::TorchDispatchModeTLS::any_modes_set() && !at::impl::torch_function_mode_enabled()) return F(args);
  } catch (const NotTaken &) {
  } catch (const std::exception &) {  // c10::Error: the general route meets and raises it again
  }
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"quantize", (PyCFunction)(void (*)())entry<quantize, 8>, METH_FASTCALL, nullptr},
    {"swiglu_quantize", (PyCFunction)(void (*)())entry<swiglu_quantize, 6>, METH_FASTCALL, nullptr},
    {"matmul", (PyCFunction)(void (*)())entry<matmul, 7>, METH_FASTCALL, nullptr},
    {"decode_step", (PyCFunction)(void (*)())entry<decode_step, 11>, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_arcq_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__arcq_host(void) {
  PyObject *m = PyModule_Create(&module);
  // (looked for in the file ahead of loading it: a library of another torch is not loaded)
  if (m && PyModule_AddStringConstant(m, "built", "built against torch " ARCQ_TORCH_VERSION) < 0) Py_CLEAR(m);
  return m;
}
